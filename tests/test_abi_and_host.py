"""CPU-side checks of the shipped pieces: the C ABI library loads and exports exactly what
include/omk_forest.h declares, errors come back as status codes, the synthetic forest
generator produces well-formed forests with the documented statistics, and the benchmark's
byte model is what it says.  No GPU compute here."""
import json
import math
import os
import re
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    text = open(os.path.join(ROOT, "include", "omk_forest.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(omk_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    import ctypes
    import omoknuni_small_amd as omk
    from omoknuni_small_amd import forest
    lib = omk.load_library()
    names = declared_functions()
    assert len(names) >= 30
    for n in names:
        assert hasattr(lib, n), "libomk_forest.so does not export " + n
    assert sorted(forest.EXPORTS) == names, "the Python mirror and the header disagree"
    assert lib.omk_version() >= 1
    assert isinstance(ctypes.c_char_p(lib.omk_last_error()).value, bytes)


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from omoknuni_small_amd import forest
    monkeypatch.setattr(forest, "_LIB", None)
    monkeypatch.setattr(forest, "_HERE", str(tmp_path))
    with pytest.raises(OSError, match="no host fallback"):
        forest.load_library()


def test_errors_are_status_codes_not_crashes():
    import omoknuni_small_amd as omk
    with pytest.raises(omk.OmkError) as e:
        omk.Forest(0)
    assert e.value.code == -1 and "capacity" in str(e.value)
    try:
        f = omk.Forest(16)
    except omk.OmkError as err:
        # no GPU in this process: creation reports the HIP failure and nothing leaks
        assert err.code == -2
        return
    f.close()


def test_bench_refuses_more_than_one_gpu():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode == 2 and "ONE GPU" in r.stderr and r.stdout == ""


def check_forest(soa, roots, meta):
    n = len(soa["N"])
    cb, cc = soa["child_begin"].astype(np.int64), soa["child_count"].astype(np.int64)
    exp = np.nonzero(cc > 0)[0]
    assert (cb[exp] >= 0).all() and (cb[exp] + cc[exp] <= n).all()
    owner = np.zeros(n, np.int32)
    for v in exp:
        owner[cb[v]:cb[v] + cc[v]] += 1
    assert owner.max() == 1, "a node has two parents"
    assert (owner[roots] == 0).all()
    legal = np.ones(n, bool)
    if soa.get("legal") is not None:
        legal = np.unpackbits(soa["legal"].view(np.uint8), bitorder="little")[:n].astype(bool)
    kids = owner == 1
    assert (soa["N"][kids & legal] >= 1).all() and (soa["N"] <= max(meta["n_cap"], soa["N"][exp].max())).all()
    assert (np.abs(soa["W"]) <= soa["N"] + 1e-3).all()
    assert (soa["VL"] == 0).all()
    for v in exp[:200]:
        sl = slice(cb[v], cb[v] + cc[v])
        lg = legal[sl]
        assert lg.any()
        assert abs(float(soa["P"][sl][lg].sum()) - 1.0) < 1e-4
        assert (soa["P"][sl][~lg] == 0).all()
        if (cc[sl] == 0).all():  # N of an expanded node was set from its children as drawn at that time
            assert soa["N"][v] == 1 + int(soa["N"][sl][lg].sum())
        assert sorted(soa["action"][sl]) == list(range(cc[v]))
    d = meta["depth"]
    assert d.max() <= meta["max_depth"] and (cc[d == meta["max_depth"]] == 0).all()
    return exp, legal


def test_synthetic_forests_are_well_formed():
    from omoknuni_small_amd import synth
    soa, roots, meta = synth.generate("c0", nodes_per_tree=30000, seed=5)
    exp, legal = check_forest(soa, roots, meta)
    assert (soa["child_count"][exp] == 225).all()
    frac = legal[soa["child_begin"][exp[0]]:][: 225 * 20].mean()
    assert 0.4 < frac < 0.6
    # same seed, same forest; another seed, another forest
    again, _, _ = synth.generate("c0", nodes_per_tree=30000, seed=5)
    assert all((soa[k] == again[k]).all() for k in soa)
    other, _, _ = synth.generate("c0", nodes_per_tree=30000, seed=6)
    assert (other["N"] != soa["N"]).any()

    soa, roots, meta = synth.generate("c2", n_trees=3, nodes_per_tree=40000, seed=5)
    exp, legal = check_forest(soa, roots, meta)
    assert list(roots) == [0, 40000, 80000]
    last = soa["child_begin"][exp] + 361
    assert legal[last].all(), "the pass move always has a child"

    soa, roots, meta = synth.generate("c3", nodes_per_tree=60000, seed=5)
    exp, _ = check_forest(soa, roots, meta)
    assert soa.get("legal") is None
    fo = soa["child_count"][exp]
    assert fo.min() >= 1 and fo.max() <= 218 and 30 < fo.mean() < 40
    for v in exp[:300]:
        p = soa["P"][soa["child_begin"][v]: soa["child_begin"][v] + soa["child_count"][v]]
        assert (np.diff(p) <= 0).all(), "children are stored by descending prior"

    soa, roots, meta = synth.generate("c4", nodes_per_tree=50000, seed=5)
    check_forest(soa, roots, meta)
    assert soa["rN"].max() <= 10000 and (np.abs(soa["rW"]) <= soa["rN"] + 1e-3).all()
    assert len(np.unique(soa["hash"])) == len(soa["hash"])


def test_zipf_statistics():
    from omoknuni_small_amd import synth
    soa, _, meta = synth.generate("c0", nodes_per_tree=120000, seed=9)
    legal = np.unpackbits(soa["legal"].view(np.uint8), bitorder="little")[: len(soa["N"])].astype(bool)
    leaves = legal & (soa["child_count"] == 0)
    leaves[0] = False
    n = soa["N"][leaves]
    # P(N = 1) = 1 / zeta(1.2), P(N >= cap) = tail mass of Zipf(1.2) beyond 10^4
    assert abs((n == 1).mean() - 1 / 5.5916) < 0.01
    assert abs((n == 2).mean() - 2 ** -1.2 / 5.5916) < 0.01
    assert abs((n == 10000).mean() - 0.142) < 0.02
    q = soa["W"][leaves] / n
    assert abs(q.mean()) < 0.02 and abs(q.std() - 1 / math.sqrt(3)) < 0.02  # uniform in [-1, 1]


def test_bench_byte_model_on_a_known_tree():
    sys.path.insert(0, ROOT)
    import bench
    # root with 3 slots (2 legal) -> child 1 expanded with 2 slots (both legal)
    soa = dict(child_begin=np.array([1, 4, 0, 0, 0, 0], np.int32), child_count=np.array([3, 2, 0, 0, 0, 0], np.int32),
               legal=np.array([0b110111], np.uint32))
    L = bench.legal_children_per_node(soa)
    assert list(L[:2]) == [2, 2]
    paths = np.array([[0, 1, 4], [0, 1, 5], [0, 3, -1]], np.int32)
    plen = np.array([3, 3, 2], np.int32)
    sel, bak, steps = bench.ByteModel(soa, {}).step(paths, plen, np.zeros(6, np.int32))
    assert steps == 5
    # per selection step: L*16 + ceil(F/8) + 24; per path entry written: 4
    assert sel == 3 * (2 * 16 + 1 + 24) + 2 * (2 * 16 + 1 + 24) + 4 * 8
    assert bak == 24 * 8 + 4 * 3 + 4 * 8
    assert list(bench.visits_of(paths, plen, 6)) == [3, 2, 0, 1, 1, 1]
    # the exact value sums of a backup: the leaf takes +v, every ply up flips the sign
    add = bench.exact_value_sums(paths, plen, np.array([0.5, -0.25, 1.0], np.float32), 6)
    assert list(add) == [0.5 - 0.25 - 1.0, -0.5 + 0.25, 0.0, 1.0, 0.5, -0.25]


def test_golden_fixture_is_data_only():
    with open(os.path.join(ROOT, "tests", "golden", "kat_reference.json")) as f:
        g = json.load(f)
    assert {"select", "score_bits", "backup", "virtual_loss_probe"} <= set(g)


def test_proof_of_non_increasing_keys_against_brute_force(tmp_path):
    """keys_provably_monotone (csrc/omk_score.h) lets the kernels skip the entry-by-entry look at a
    child's successive scores; on the host, with the same arithmetic, every "proven" case is
    evaluated entry by entry (tests/cpp/lemma_check.cpp), and the test must say yes often enough
    to be worth having."""
    import re
    import subprocess
    exe = str(tmp_path / "lemma_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", "-I",
                           os.path.join(ROOT, "omoknuni_small_amd", "csrc"),
                           os.path.join(ROOT, "tests", "cpp", "lemma_check.cpp"), "-o", exe])
    out = subprocess.run([exe, "200000"], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout[-2000:]
    m = re.search(r"provably monotone: (\d+) without RAVE, (\d+) with; counter-examples 0", out.stdout)
    assert m, out.stdout[-500:]
    assert int(m.group(1)) > 100000 and int(m.group(2)) > 100000


def test_merge_rules_against_the_serial_loop(tmp_path):
    """The rules by which the selection kernels settle a node whose visitors split (a root's block up to 64 of them, the
    helpers of a team any number), restated step by step on the host with the kernels' own score arithmetic
    (tests/cpp/merge_check.cpp): every node they accept must come out as the serial loop plays it."""
    import re
    import subprocess
    exe = str(tmp_path / "merge_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", "-I",
                           os.path.join(ROOT, "omoknuni_small_amd", "csrc"),
                           os.path.join(ROOT, "tests", "cpp", "merge_check.cpp"), "-o", exe])
    out = subprocess.run([exe, "60000", "7"], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout[-2000:]
    m = re.search(r"blocks: merged (\d+), declined \d+; teams: merged (\d+), declined \d+; wrong 0", out.stdout)
    assert m and int(m.group(1)) > 30000 and int(m.group(2)) > 30000, out.stdout[-500:]
    m = re.search(r"lists cut short: (\d+)", out.stdout)
    assert m and int(m.group(1)) > 30, out.stdout[-500:]


def test_bounds_of_scores_hold_the_exact_ones(tmp_path):
    """Children are ruled out by bounds worked out with approximate reciprocals (score_about): over the whole range of counts,
    sums, priors and blends, with reciprocals off by two units in the last place either way, the exact score lies between them
    (tests/cpp/bound_check.cpp)."""
    import re
    import subprocess
    exe = str(tmp_path / "bound_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", "-I",
                           os.path.join(ROOT, "omoknuni_small_amd", "csrc"),
                           os.path.join(ROOT, "tests", "cpp", "bound_check.cpp"), "-o", exe])
    out = subprocess.run([exe, "1000000"], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout[-2000:]
    m = re.search(r"bounds: (\d+) held, wrong 0", out.stdout)
    assert m and int(m.group(1)) > 1800000, out.stdout[-500:]


def test_tickets_are_drawn_between_barriers_of_the_wavefront():
    """Lane 0 draws a wavefront's next ticket at the head of loops that may end in another branch of lane 0's own.  Without a
    barrier of the wavefront the compiler may join the two across the loop's edge, and the other lanes go round without the
    ticket: every loop draws through the one function that has them (take_ticket)."""
    import re
    csrc = os.path.join(ROOT, "omoknuni_small_amd", "csrc")
    text = ""
    for name in ("omk_select_kernels.h", "omk_select_blocks.h"):
        with open(os.path.join(csrc, name)) as f:
            text += f.read()
    body = re.search(r"int take_ticket\(.*?\n}\n", text, re.S).group(0)
    assert re.search(r"wave_barrier\(\);\s*if \(lane == 0\) ticket = atomicAdd\(counter, 1\);\s*__builtin_amdgcn_wave_barrier\(\);", body)
    assert not re.search(r"atomicAdd\(\s*&?[\w.>-]*\b(head|next|sched_head|singles_head)\s*,", text)
    assert len(re.findall(r"= take_ticket\(", text)) == 4


def test_loads_of_a_node_are_waited_for_where_they_are_made():
    """A wavefront of a block asks for a node's children in two places.  Loads that are not known done where its loop comes
    round make the compiler wait in front of the next node's, and for the stores of the level before with them: all of
    them are waited for (vmcnt 0), in both places, before anything but what may overlap with them."""
    import re
    with open(os.path.join(ROOT, "omoknuni_small_amd", "csrc", "omk_select_blocks.h")) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    asked = re.findall(r"\n\s*ask\(\);(.*?)__builtin_amdgcn_s_waitcnt\(0x0F70\);", text, re.S)
    assert len(asked) == 2 and len(re.findall(r"\bask\(\);", text)) == 2
    assert not any(re.search(r"\bk\.|\bsp\[|\bword\[", between) for between in asked)


def test_stores_for_other_blocks_are_waited_for_by_who_made_them():
    """A helper's stores that its owner, or another helper, announces to other blocks with a release of agent scope: that
    release waits for the announcing wavefront's own stores, a release of workgroup scope and a block barrier for none in
    memory.  The helper waits before it says that it is done."""
    import re
    with open(os.path.join(ROOT, "omoknuni_small_amd", "csrc", "omk_select_kernels.h")) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    body = lambda name: re.search(r"void %s\(.*?\n}\n" % name, text, re.S).group(0)
    before = r"wait_stores\(\);\s*"
    assert re.search(before + r'__builtin_amdgcn_fence\(__ATOMIC_RELEASE, "workgroup"\);\s*if \(lane == 0\) atomicAdd\(&pl.finished',
                     body("partition_chunks"))
    assert re.search(r"if \(goff >= 0\) " + before + r"__syncthreads\(\);\s*}\s*$", body("team_merge"))
    helpers = body("k_select_groups").split("for (;;)", 1)[1]
    assert len(re.findall(r"if \(HEAVY\) " + before + r"__syncthreads\(\);", helpers)) == 2


def test_staging_is_not_handed_out_over_what_kernels_still_read(tmp_path):
    """The pinned block's staging (csrc/omk_staging.h) against a stream that runs as late as it can
    (tests/cpp/staging_check.cpp): after a wrap, an offset that was in use before says nothing about what
    has run."""
    exe = str(tmp_path / "staging_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", os.path.join(ROOT, "tests", "cpp", "staging_check.cpp"),
                           "-o", exe])
    out = subprocess.run([exe, "3000"], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok 3000\n", out.stdout


@pytest.mark.parametrize("n", [0, 1, 300_000, 2_097_152, 2_097_153, 5_000_000])
def test_one_downloaded_array_does_not_keep_a_large_tree_alive(n):
    from omoknuni_small_amd import forest
    got = forest._together(n, N=np.int32, W=np.float32, P=np.float32, VL=np.int32)
    for k, a in got.items():
        assert a.shape == (n,) and a.dtype == (np.float32 if k in "WP" else np.int32) and a.flags["C_CONTIGUOUS"]
        owner = a
        while owner.base is not None:
            owner = owner.base
        assert owner.nbytes <= max(32 << 20, a.nbytes)


def test_no_exception_crosses_the_c_boundary():
    """More nodes than a host vector can hold: a status, not an abort (in a process of its own, should it be one)."""
    program = """
import ctypes as C
import numpy as np
from omoknuni_small_amd import forest as F
lib = F.load_library()
a = dict(N=np.zeros(4, np.int32), W=np.zeros(4, np.float32), P=np.zeros(4, np.float32), VL=np.zeros(4, np.int32), rN=None,
         rW=None, child_begin=np.zeros(4, np.int32), child_count=np.zeros(4, np.int32), action=None, legal=None, hash=None)
v = F._view_of(a)
v.n_nodes = 1 << 61
i, f = F._ptr(a["N"], F.i32p), F._ptr(a["W"], F.f32p)
none = C.c_void_p()
print(lib.omk_soa_compact_legal(C.byref(v), C.c_int64(4), i, f, f, i, none, none, i, i, none, none, none, none),
      lib.omk_last_error().decode())
"""
    r = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True, cwd=ROOT)
    assert r.returncode == 0 and r.stdout.startswith("-1 out of host memory"), (r.returncode, r.stdout, r.stderr[-500:])
