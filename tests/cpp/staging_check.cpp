// The staging bookkeeping (omk_staging.h) against a stream that runs as late as it can: calls stage a piece that one
// enqueued kernel reads, now and then one waits, and some remember a point of the stream and later learn that it has
// been reached.  No piece may be handed out over one whose reader has not run.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../omoknuni_small_amd/csrc/omk_staging.h"

struct Piece {
    size_t at, end;
};

// The bookkeeping under test with the stream behind it.
struct Model {
    omk::Staging staging;
    std::vector<Piece> unread;  // pieces of kernels that have not run, in the order of the stream
    explicit Model(size_t room) : staging(room) {}

    bool stage(size_t bytes) {
        size_t at = staging.take(bytes);
        if (at == omk::Staging::kFull) {  // the caller waits for the stream and starts over
            unread.clear();
            staging.idle();
            at = staging.take(bytes);
            if (at == omk::Staging::kFull) return false;
        }
        const size_t end = at + bytes;
        if (at % 128 != 0 || end > staging.room()) return false;
        for (const Piece &p : unread)
            if (at < p.end && p.at < end) return false;
        unread.push_back({at, end});
        return true;
    }
};

int main(int argc, char **argv) {
    const int runs = argc > 1 ? atoi(argv[1]) : 2000;
    {  // a point of the stream, a wrap, the same offset again: the pieces behind the wrap are still to be read
        Model m(4 << 20);
        if (!m.stage(2400000)) return 1;
        const uint64_t point = m.staging.now();
        if (!m.stage(2400000)) return 1;  // does not fit: waits, and starts at the front
        m.staging.ran_to(point);          // reached long ago, and says nothing about the piece behind it
        if (!m.stage(256)) return printf("the piece behind the wrap was written over\n"), 1;
    }
    {  // nothing handed out since: the front again
        Model m(4096);
        if (!m.stage(1000)) return 1;
        const uint64_t point = m.staging.now();
        m.unread.clear();
        m.staging.ran_to(point);
        if (m.staging.take(4096) != 0) return printf("staging was not given back\n"), 1;
    }
    std::mt19937 rng(7);
    for (int r = 0; r < runs; r++) {
        Model m(128 * (1 + rng() % 40));
        uint64_t point = 0;
        size_t before = 0;  // pieces unread when the point was taken that are unread still
        bool marked = false;
        for (int step = 0; step < 200; step++) {
            switch (rng() % 8) {
                case 0:  // a call that waits for the stream
                    m.unread.clear();
                    m.staging.idle();
                    before = 0;
                    break;
                case 1:
                    point = m.staging.now();
                    before = m.unread.size();
                    marked = true;
                    break;
                case 2:  // the stream has got to the point, and no further
                    if (!marked) break;
                    m.unread.erase(m.unread.begin(), m.unread.begin() + before);
                    before = 0;
                    m.staging.ran_to(point);
                    break;
                default: {
                    const size_t had = m.unread.size();
                    if (!m.stage(1 + rng() % m.staging.room())) return printf("run %d step %d\n", r, step), 1;
                    if (m.unread.size() <= had) before = 0;  // it waited on the way
                }
            }
        }
    }
    printf("ok %d\n", runs);
    return 0;
}
