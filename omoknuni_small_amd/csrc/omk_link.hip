// Bulk transfers between the host's arrays and the forest's through the pinned block: the words of up to
// kMaxSegments arrays, one array after the other, are one stream that is cut into pieces; a piece is copied to
// or from pinned memory by the host and spread or collected by one kernel.
#include "omk_internal.h"

namespace omk {

// Which array word i of the stream belongs to, and where it lies on the device.
__device__ __forceinline__ uint32_t *segment_word(const Segments &g, int64_t i) {
    int q = 0;
    while (q + 1 < g.n && i >= g.start[q + 1]) q++;
    return g.dev[q] + (i - g.start[q]) * g.step[q];
}

// Four words per thread, a wavefront's worth apart: what bounds both kernels is the host link, and four trips in
// flight per lane fill it (reads 41 GB/s, writes 50 GB/s of the copy engine's 53 in pieces of 4 MB).
constexpr int kPieceWords = 1024;

__global__ __launch_bounds__(256) void k_put(Segments g, const uint32_t *staged, int64_t first, int64_t count,
                                             HostSignal sig) {
    const int64_t base = (int64_t)blockIdx.x * kPieceWords + threadIdx.x;
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (base + 256 * j < count) v[j] = staged[base + 256 * j];
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (base + 256 * j < count) *segment_word(g, first + base + 256 * j) = v[j];
    if (sig.flag) host_signal(sig.count, sig.flag, sig.seq, gridDim.x);
}

__global__ __launch_bounds__(256) void k_get(Segments g, uint32_t *staged, int64_t first, int64_t count, HostSignal sig) {
    const int64_t base = (int64_t)blockIdx.x * kPieceWords + threadIdx.x;
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (base + 256 * j < count) v[j] = *segment_word(g, first + base + 256 * j);
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (base + 256 * j < count) host_store(staged + base + 256 * j, v[j]);
    host_signal(sig.count, sig.flag, sig.seq, gridDim.x);
}

hipError_t launch_put(const Segments &g, const uint32_t *staged, int64_t first, int64_t count, const HostSignal &sig,
                      hipStream_t s) {
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_put, dim3((unsigned)((count + kPieceWords - 1) / kPieceWords)), dim3(256), 0, s, g, staged, first,
                       count, sig);
    return hipGetLastError();
}

hipError_t launch_get(const Segments &g, uint32_t *staged, int64_t first, int64_t count, const HostSignal &sig,
                      hipStream_t s) {
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_get, dim3((unsigned)((count + kPieceWords - 1) / kPieceWords)), dim3(256), 0, s, g, staged, first,
                       count, sig);
    return hipGetLastError();
}

}  // namespace omk
