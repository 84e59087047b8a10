"""What crosses between the host and the card through pinned memory: leaf gather, roots, values, offers, keys.
At the sizes where the kernels that carry it can go wrong (edges of their tiles), against the CPU checker."""
import numpy as np
import pytest

from oracle import ref_cpu as R
from tests.helpers import random_tree

pytestmark = pytest.mark.gpu


def mapped():
    """The process's mappings of device and pinned memory."""
    with open("/proc/self/maps") as lines:
        return {line.split()[0] for line in lines if "/dev/" in line}


# the gather takes 64 traversals x 32 depths at a time (a path has one node more than the depth bound)
@pytest.mark.parametrize("depth", [1, 30, 31, 32, 33, 70])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 300])
def test_leaf_gather_at_the_edges_of_its_tiles(n, depth):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(5 + n, n_expand=300, fanout=(1, 5), max_depth=60, n_roots=3)
    ref = R.RefTree.from_soa(soa)
    troots = roots[np.arange(n) % 3]
    f = omk.Forest.from_soa(soa)
    b = omk.Batch(f, n, depth)
    rng = np.random.default_rng(n)
    b.set_roots(troots)
    for _ in range(3):
        rpaths, rlen, rleaf, _ = ref.select_batch(troots, R.make_params(c_puct=1.4, virtual_loss=3, max_depth=depth))
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        paths, plen, leaf, actions = b.read()
        assert (paths == rpaths).all() and (plen == rlen).all() and (leaf == rleaf).all()
        assert (actions == ref.gather_actions(rpaths, rlen)).all()
        values = (rng.integers(-64, 65, n) / 64.0).astype(np.float32)
        ref.backup_batch(rpaths, rlen, values, 3)
        b.set_values(values)
        b.backup(3)
        ref.W[:] = f.download()["W"]


# roots in any order, with and without crowds: the grouping is a radix sort of eleven bits a pass
@pytest.mark.parametrize("n,n_roots,shuffled", [(2, 1, False), (5, 5, True), (64, 64, False), (500, 7, True), (3000, 2100, True)])
def test_roots_in_any_order(n, n_roots, shuffled):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(n, n_expand=2 * n_roots, fanout=(1, 6), max_depth=5, n_roots=n_roots)
    troots = roots[np.arange(n) % n_roots]
    if shuffled:
        troots = np.random.default_rng(n).permutation(troots)
    ref = R.RefTree.from_soa(soa)
    f = omk.Forest.from_soa(soa)
    b = omk.Batch(f, n + 10, 6)
    for use in (troots, troots[::-1][:max(1, n // 2)]):
        rpaths, rlen, rleaf, _ = ref.select_batch(use, R.make_params(c_puct=1.4, virtual_loss=3, max_depth=6))
        b.set_roots(use)
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        paths, plen, leaf, _ = b.read()
        assert (paths == rpaths).all() and (plen == rlen).all() and (leaf == rleaf).all()


# one thread per child, 256 a round; leaves known from a read, from none, and from one that a backup has overtaken
@pytest.mark.parametrize("moves", [1, 255, 256, 257, 1000])
def test_expansion_after_a_read_and_without(moves):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(11, n_expand=30, fanout=(2, 6), max_depth=4, n_roots=2, vl_frac=0.0)
    ref = R.RefTree.from_soa(soa)
    n, A = 24, 1003
    troots = roots[np.arange(n) % 2]
    f = omk.Forest.from_soa(soa, capacity=ref.n + 3 * n * moves)
    b = omk.Batch(f, n, 8)
    b.set_roots(troots)
    rng = np.random.default_rng(moves)
    for step in range(3):
        rpaths, rlen, rleaf, _ = ref.select_batch(troots, R.make_params(c_puct=1.4, virtual_loss=3, max_depth=8))
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        if step != 1:
            assert (b.read()[2] == rleaf).all()
        counts = np.where(rng.random(n) < 0.3, 0, moves)
        begin = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
        mv = np.concatenate([rng.permutation(A + 2)[:c] for c in counts] + [[]]).astype(np.int32)  # two outside
        policy = rng.uniform(-0.2, 1.2, (n, A)).astype(np.float32)
        values = (rng.integers(-64, 65, n) / 64.0).astype(np.float32)
        widening = (2.0, 0.5) if step == 2 else None
        if step == 2:  # the widening then has to see the visits of this backup
            ref.backup_batch(rpaths, rlen, values, 3)
            b.set_values(values)
            b.backup(3)
        want = ref.expand_batch(rleaf, begin, mv, policy=policy, action_space=A, widening=widening)
        got = b.expand_ex(begin, mv, (np.arange(n + 1) * A).astype(np.int32), policy, A, widening=widening)
        assert (got == want).all()
        if step != 2:
            ref.backup_batch(rpaths, rlen, values, 3)
            b.set_values(values)
            b.backup(3)
        st, sx = f.download(), f.download_structure()
        ref.W[:] = st["W"]
        assert (st["N"] == ref.N).all() and st["P"].tobytes() == ref.P.tobytes() and (st["VL"] == ref.VL).all()
        assert (sx["child_begin"] == ref.child_begin).all() and (sx["child_count"] == ref.child_count).all()
        assert (sx["action"] == ref.action).all()


# one block serves a root: up to 1024 slots, ranks from the ballots of 16 wavefronts
@pytest.mark.parametrize("slots,mask_frac", [(1, 0.0), (64, 0.0), (65, 0.4), (1024, 0.0), (1024, 0.5)])
def test_root_queries_at_every_width(slots, mask_frac):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(slots, n_expand=1, fanout=(slots, slots), max_depth=1, mask_frac=mask_frac, n_max=90)
    ids = np.arange(1, slots + 1)
    legal = ids if not mask_frac else ids[((soa["legal"][ids >> 5] >> (ids & 31).astype(np.uint32)) & 1) == 1]
    f = omk.Forest.from_soa(soa)
    gamma = np.random.default_rng(slots).gamma(0.3, 1.0, len(legal)).astype(np.float32)
    with pytest.raises(omk.OmkError):
        f.add_root_noise(0, np.append(gamma, gamma[:1]), 0.25)
    assert f.download()["P"].tobytes() == soa["P"].tobytes()
    f.add_root_noise(0, gamma, 0.25)
    total = np.float32(0.0)
    for g in gamma:
        total = np.float32(total + g)
    want = soa["P"].copy()
    want[legal] = np.float32(0.75) * want[legal] + np.float32(0.25) * (gamma / total)
    assert f.download()["P"].tobytes() == want.tobytes()
    probs, n = f.action_probabilities(0, 0.0, slots)
    best = legal[np.argmax(soa["N"][legal])]
    assert n == len(legal) and np.flatnonzero(probs).tolist() == [soa["action"][best]]
    assert f.reroot_child(0, int(soa["action"][legal[-1]])) == legal[-1] and f.reroot_child(0, slots) == -1


# arrays cross as one stream of words, in pieces of 2^18, four on their way at a time
@pytest.mark.parametrize("n", [1, 37, 43690, 43691, 200_001])
@pytest.mark.parametrize("rave", [False, True])
def test_arrays_cross_in_pieces(n, rave):
    import omoknuni_small_amd as omk
    rng = np.random.default_rng(n)
    fan = rng.integers(1, 9, n)
    soa = dict(N=rng.integers(0, 999, n).astype(np.int32), W=rng.random(n).astype(np.float32),
               P=rng.random(n).astype(np.float32), VL=rng.integers(0, 9, n).astype(np.int32),
               child_begin=np.zeros(n, np.int32), child_count=np.zeros(n, np.int32),
               action=rng.integers(0, 400, n).astype(np.int32), hash=rng.integers(0, 1 << 63, n).astype(np.uint64))
    at, node = 1, 0
    while at < n and node < at:
        k = int(min(fan[node], n - at))
        soa["child_begin"][node], soa["child_count"][node] = at, k
        at, node = at + k, node + int(rng.integers(1, 3))
    if rave:
        soa.update(rN=rng.integers(0, 99, n).astype(np.int32), rW=rng.random(n).astype(np.float32))
    f = omk.Forest.from_soa(soa, capacity=n + 5)
    for scale in (1, 2):
        soa["W"] = soa["W"] * np.float32(scale)
        f.upload(soa)
        got = dict(f.download(), **f.download_structure())
        for k in got:
            assert got[k].tobytes() == soa[k].tobytes(), k


@pytest.mark.parametrize("fault,message", [("two parents", "two parents"), ("own child", "own child"), ("outside", "outside"),
                                           ("negative", "< 0"), ("wide", "exceeds")])
def test_structures_that_are_no_forest_are_refused(fault, message):
    import omoknuni_small_amd as omk
    n = 5000
    soa = dict(N=np.ones(n, np.int32), W=np.zeros(n, np.float32), P=np.zeros(n, np.float32), VL=np.zeros(n, np.int32),
               child_begin=np.zeros(n, np.int32), child_count=np.zeros(n, np.int32))
    soa["child_begin"][[0, 70, 133]], soa["child_count"][[0, 70, 133]] = [1, 100, 1003], [64, 903, 1]
    f = omk.Forest.from_soa(soa)
    before = f.download_structure()
    bad = dict(soa, child_begin=soa["child_begin"].copy(), child_count=soa["child_count"].copy())
    bad["child_begin"][199], bad["child_count"][199] = {"two parents": (1002, 3), "own child": (199, 1), "outside": (n - 1, 2),
                                                        "negative": (3, -1), "wide": (1100, 1025)}[fault]
    with pytest.raises(omk.OmkError, match=message):
        f.upload(bad)
    after = f.download_structure()
    assert all((before[k] == after[k]).all() for k in before)


# 256 blocks share a level and write 64 nodes' children at a time; twelve levels are enqueued before the host looks
@pytest.mark.parametrize("shape", ["chain of 40", "one level of 1000", "wide levels", "a leaf"])
@pytest.mark.parametrize("static", [False, True])
def test_compaction_of_every_shape(shape, static):
    import omoknuni_small_amd as omk
    rng = np.random.default_rng(len(shape))
    counts = {"chain of 40": [1] * 40, "one level of 1000": [1000], "a leaf": [3],
              "wide levels": [200] + [int(x) for x in rng.integers(0, 60, 200)] + [int(x) for x in rng.integers(0, 9, 3000)]}[shape]
    n = 1 + sum(counts) + 17
    begin, count = np.zeros(n, np.int32), np.zeros(n, np.int32)
    at = 1
    for node, c in enumerate(counts):
        if node < at and c:
            begin[node], count[node] = at, c
            at += c
    soa = dict(N=rng.integers(0, 99, n).astype(np.int32), W=rng.random(n).astype(np.float32), P=rng.random(n).astype(np.float32),
               VL=rng.integers(0, 5, n).astype(np.int32), child_begin=begin, child_count=count,
               action=rng.integers(0, 99, n).astype(np.int32), legal=rng.integers(0, 1 << 32, (n + 31) // 32).astype(np.uint32),
               hash=rng.integers(0, 1 << 63, n).astype(np.uint64), rN=rng.integers(0, 9, n).astype(np.int32),
               rW=rng.random(n).astype(np.float32))
    root = 2 if shape == "a leaf" else 0
    f = omk.Forest.from_soa(soa)
    order = f.compact(root, static=static)
    ref, want = R.RefTree.from_soa(soa).compacted(root)
    assert (order == want).all()
    got = dict(f.download(), **f.download_structure())
    for k in ("N", "W", "P", "VL", "rN", "rW", "action"):
        assert got[k].tobytes() == soa[k][order].tobytes(), k
    assert (got["child_begin"] == ref.child_begin).all() and (got["child_count"] == ref.child_count).all()


# trees whose arrays do not all fit the scratch at once: two rounds, and an array at a time
@pytest.mark.parametrize("fan", [500, 1399])
def test_compaction_of_large_trees(fan):
    import omoknuni_small_amd as omk
    rng = np.random.default_rng(fan)
    upper = 1 + 3 + 3000  # the root, its children, theirs; `fan` children each of the latter, in falling order
    n = upper + 3000 * fan
    begin, count = np.zeros(n, np.int32), np.zeros(n, np.int32)
    if fan > 1024:  # (two levels in the place of one)
        wide = np.array([700, fan - 700])
        n = upper + 3000 * 2 + 3000 * fan
        begin, count = np.zeros(n, np.int32), np.zeros(n, np.int32)
    begin[0], count[0] = 1, 3
    begin[1:4], count[1:4] = 4 + 1000 * np.arange(3)[::-1], 1000
    second = np.arange(4, upper)
    levels = [np.array([0]), np.arange(1, 4), np.concatenate([np.arange(b, b + 1000) for b in begin[1:4]])]
    if fan > 1024:
        begin[second], count[second] = upper + 2 * np.arange(3000)[::-1], 2
        third = np.arange(upper, upper + 6000)
        count[third] = np.tile(wide, 3000)
        begin[third] = upper + 6000 + np.concatenate([[0], np.cumsum(count[third])[:-1]])
    else:
        begin[second], count[second] = upper + fan * np.arange(3000)[::-1], fan
    while count[levels[-1]].any():
        up = levels[-1][count[levels[-1]] > 0]
        step = np.repeat(begin[up] - np.concatenate([[0], np.cumsum(count[up])[:-1]]), count[up])
        levels.append(step + np.arange(len(step)))
    order = np.concatenate(levels)
    assert len(order) == n
    new_id = np.empty(n, np.int32)
    new_id[order] = np.arange(n)
    soa = dict(N=rng.integers(0, 99, n).astype(np.int32), W=rng.random(n).astype(np.float32), P=rng.random(n).astype(np.float32),
               VL=rng.integers(0, 5, n).astype(np.int32), child_begin=begin, child_count=count,
               action=rng.integers(0, 99, n).astype(np.int32), hash=rng.integers(0, 1 << 63, n).astype(np.uint64),
               rN=rng.integers(0, 9, n).astype(np.int32), rW=rng.random(n).astype(np.float32))
    f = omk.Forest.from_soa(soa)
    assert (f.compact(0) == order).all()
    got = dict(f.download(), **f.download_structure())
    for k in ("N", "W", "P", "VL", "rN", "rW", "action"):
        assert got[k].tobytes() == soa[k][order].tobytes(), k
    assert (got["child_count"] == count[order]).all()
    inner = count[order] > 0
    assert (got["child_begin"][inner] == new_id[begin[order][inner]]).all()
    # the keys have come along: a table filled by the new ids finds the leaves by them
    table = omk.TranspositionTable(f, 12)
    b = omk.Batch(f, 500, 5)
    b.set_roots(np.zeros(500, np.int32))
    b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
    leaf = np.unique(b.read()[2])
    table.insert(soa["hash"][order[leaf]], leaf)
    assert (table.probe_leaves(b) == b.read()[2]).all()


# a young tree: the visitors spread over children without visits, whose first entries are nearly all of the merge that the
# root's block makes, or beyond 64 visitors or 384 children the helpers of a team
@pytest.mark.parametrize("children", [65, 130, 225, 362, 700])
@pytest.mark.parametrize("n", [8, 23, 63, 64, 65])
@pytest.mark.parametrize("rave", [False, True])
def test_visitors_spread_over_a_fresh_node(children, n, rave):
    import omoknuni_small_amd as omk
    soa = dict(N=np.zeros(1, np.int32), W=np.zeros(1, np.float32), P=np.ones(1, np.float32), VL=np.zeros(1, np.int32),
               child_begin=np.zeros(1, np.int32), child_count=np.zeros(1, np.int32), action=np.full(1, -1, np.int32))
    if rave:
        soa.update(rN=np.zeros(1, np.int32), rW=np.zeros(1, np.float32))
    ref = R.RefTree.from_soa(soa)
    f = omk.Forest.from_soa(soa, capacity=1 + children * (1 + 3 * n))
    b = omk.Batch(f, n, 6)
    b.enable_stats()
    rng = np.random.default_rng(children + n)
    spread, teams = 0, n > 64 or children > 384
    for step in range(4):
        k = 1 if step == 0 else n
        roots = np.zeros(k, np.int32)
        rpaths, rlen, rleaf, _ = ref.select_batch(roots, R.make_params(c_puct=1.4, virtual_loss=3, use_rave=rave, rave_k=1000.0,
                                                                       max_depth=6))
        b.set_roots(roots)
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3, use_rave=rave, rave_k=1000.0))
        paths, plen, leaf, _ = b.read()
        assert (paths == rpaths).all() and (plen == rlen).all() and (leaf == rleaf).all(), step
        st = b.stats()
        spread += st["merged_by_teams" if teams else "merged_by_blocks"]
        assert st["merged_by_blocks" if teams else "merged_by_teams"] == 0, st
        begin = (np.arange(k + 1) * children).astype(np.int32)
        moves = np.tile(np.arange(children, dtype=np.int32), k)
        policy = rng.random((k, children)).astype(np.float32)
        policy = np.round(policy * 50) / 50 if step == 2 else policy  # ties
        ref.expand_batch(rleaf, begin, moves, policy=policy, action_space=children)
        b.expand(begin, moves, policy=policy.astype(np.float32), action_space=children)
        values = (rng.integers(-64, 65, k) / 64.0).astype(np.float32)
        ref.backup_batch(rpaths, rlen, values, 3)
        b.set_values(values)
        b.backup(3)
    assert (f.download()["N"] == ref.N).all()
    if not rave and n >= 23:
        assert spread > 0


# settling a batch: 256 traversals share a table of their nodes; with a root each nothing is atomic
@pytest.mark.parametrize("n,n_roots", [(1, 1), (255, 1), (257, 3), (40, 40), (300, 300)])
@pytest.mark.parametrize("vl", [3, 0])
@pytest.mark.parametrize("how", ["backup", "revert"])
def test_settling_a_batch(n, n_roots, vl, how):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(n, n_expand=3 * n_roots + 20, fanout=(1, 6), max_depth=6, n_roots=n_roots, vl_frac=0.4)
    troots = roots[np.arange(n) % n_roots]
    ref = R.RefTree.from_soa(soa)
    f = omk.Forest.from_soa(soa)
    b = omk.Batch(f, n, 7)
    b.set_roots(troots)
    values = (np.random.default_rng(n).integers(-64, 65, n) / 64.0).astype(np.float32)
    b.set_values(values)
    for _ in range(2):
        rpaths, rlen, _, _ = ref.select_batch(troots, R.make_params(c_puct=1.4, virtual_loss=vl, max_depth=7))
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=vl))
        if how == "backup":
            ref.backup_batch(rpaths, rlen, values, vl)
            b.backup(vl)
        else:
            ref.revert_vl_paths(rpaths, rlen, vl)
            b.revert_vl(vl)
        got = f.download()
        assert (got["N"] == ref.N).all() and (got["VL"] == ref.VL).all()
        err = np.abs(got["W"].astype(np.float64) - ref.W) / np.maximum(np.abs(ref.W), 1.0)
        assert err.max() <= 1e-5
        ref.W[:] = got["W"]


# set_roots makes the next selection's reset; one without new roots, one whose number has been changed since and one
# with statistics make their own
@pytest.mark.parametrize("n,n_roots", [(2, 1), (256, 3), (257, 250), (1500, 1)])
def test_selections_after_set_roots_and_without(n, n_roots):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(n, n_expand=2 * n_roots + 60, fanout=(1, 6), max_depth=6, n_roots=n_roots)
    troots = roots[np.arange(n) % n_roots]
    ref = R.RefTree.from_soa(soa)
    f = omk.Forest.from_soa(soa)
    b = omk.Batch(f, n, 7)
    for step in range(7):
        rpaths, rlen, _, _ = ref.select_batch(troots, R.make_params(c_puct=1.4, virtual_loss=3, max_depth=7))
        if step not in (1, 4):
            b.set_roots(troots)
        if step == 2:
            b.debug_set_select_count(1000)
        if step == 3:
            b.debug_set_select_count((1 << 30) - 3)
        b.enable_stats(step == 5)
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        paths, plen, _, _ = b.read()
        assert (paths == rpaths).all() and (plen == rlen).all()
        ref.revert_vl_paths(rpaths, rlen, 3)
        b.revert_vl(3)


# the noise of a root that the expansion before has given its children, of another node, and after an upload
@pytest.mark.parametrize("moves", [1, 63, 64, 257])
def test_root_noise_after_an_expansion(moves):
    import omoknuni_small_amd as omk
    n = 5
    zeros = np.zeros(n, np.int32)
    soa = dict(N=zeros, W=np.zeros(n, np.float32), P=np.ones(n, np.float32), VL=zeros, child_begin=zeros,
               child_count=zeros, action=zeros - 1)
    f = omk.Forest.from_soa(soa, capacity=n * (2 * moves + 1))
    b = omk.Batch(f, n, 4)
    rng = np.random.default_rng(moves)
    gamma = rng.gamma(0.3, 1.0, moves).astype(np.float32)
    total = np.float32(0)
    for g in gamma:
        total = total + g
    noise = gamma / total if total > 0 else np.full(moves, np.float32(1) / np.float32(moves))
    begin = (np.arange(n + 1) * moves).astype(np.int32)
    b.set_roots(np.arange(n, dtype=np.int32))
    for step in range(2):  # the second expansion is that of a child of each root
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        first = b.expand(begin, np.tile(np.arange(moves, dtype=np.int32), n))
        b.revert_vl(3)
        for root in (1, 3):
            with pytest.raises(omk.OmkError, match="samples"):
                f.add_root_noise(root, np.append(gamma, gamma[:1]), 0.25)
            before = f.download()["P"]
            f.add_root_noise(root, gamma, 0.25)
            begins = f.download_structure()["child_begin"][root]
            want = before.copy()
            mine = slice(begins, begins + moves)
            want[mine] = (np.float32(1) - np.float32(0.25)) * before[mine] + np.float32(0.25) * noise
            assert (f.download()["P"] == want).all()
    assert len(first) == n


# eight moves at a time and the rest one by one; values that the clamp changes, moves outside the action space
@pytest.mark.parametrize("moves", list(range(1, 18)) + [225])
def test_priors_from_a_policy(moves):
    import omoknuni_small_amd as omk
    zeros = np.zeros(1, np.int32)
    soa = dict(N=zeros, W=np.zeros(1, np.float32), P=np.ones(1, np.float32), VL=zeros, child_begin=zeros,
               child_count=zeros, action=zeros - 1)
    f = omk.Forest.from_soa(soa, capacity=1 + moves)
    b = omk.Batch(f, 1, 4)
    b.set_roots([0])
    b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
    A = 300
    rng = np.random.default_rng(moves)
    policy = (rng.standard_normal(A) * 2).astype(np.float32)
    policy[rng.integers(0, A, 90)] = np.repeat(np.float32([np.nan, np.inf, -np.inf, -0.0, 1.0, 0.0]), 15)
    mv = rng.integers(-3, A + 3, moves).astype(np.int32)
    b.expand_ex([0, moves], mv, [0, A], policy, A)
    value = policy[np.clip(mv, 0, A - 1)]
    with np.errstate(invalid="ignore"):
        want = np.where(value > 0, np.where(value < 1, value, np.float32(1)), np.float32(0))
    want = np.where((mv >= 0) & (mv < A), want, np.float32(0.01)).astype(np.float32)
    got = f.download()["P"][1:]
    assert (got.view(np.int32) == want.view(np.int32)).all()
    assert (f.download_structure()["action"][1:] == mv).all()


# hits straight to the host, with the counts up to a megabyte and after them beyond: the same as on the device
@pytest.mark.parametrize("n,depth", [(1, 1), (51, 5), (64, 4), (513, 7), (262144 // 8, 8), (262144 // 8 + 1, 8)])
def test_table_hits_on_the_host_and_on_the_device(n, depth):
    import ctypes as C
    import omoknuni_small_amd as omk
    soa, roots = random_tree(n, n_expand=400, fanout=(2, 6), max_depth=9, n_roots=3)
    soa = dict(soa, hash=np.random.default_rng(n).integers(1, 60, len(soa["N"])).astype(np.uint64))
    got = []
    for direct in (True, False):
        f = omk.Forest.from_soa(soa)
        b = omk.Batch(f, n, depth)
        table = omk.TranspositionTable(f, 12)
        b.set_roots(roots[np.arange(n) % 3])
        for _ in range(2):
            b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
            if direct:
                hits, counts = table.traverse(b)
            else:
                hits, words = np.empty((n, depth), np.int32), np.zeros(4, np.int32)
                buf = f.dev_alloc(hits.nbytes)
                assert f._lib.omk_tt_traverse(table._h, b._h, None, 0, None, None, None, C.c_void_p(buf),
                                              words.ctypes.data_as(C.c_void_p)) == 0
                f.d2h(hits, buf)
                f.dev_free(buf)
                counts = tuple(words.tolist())
            got.append((hits, counts))
            b.backup(3)
    for a, b in zip(got[:2], got[2:]):
        assert (a[0] == b[0]).all() and a[1] == b[1]
    assert n == 1 or (got[1][0] >= 0).any()


# one traversal per tree, read every time: from the second selection on the walkers send their own rows (up to 1024
# traversals and a depth bound of 63), which a read finds after whatever was staged in between, twice if it asks
# twice, and not once a backup has changed what they say
@pytest.mark.parametrize("n,depth", [(1, 5), (3, 1), (4, 63), (5, 64), (257, 8), (1024, 6), (1025, 6)])
@pytest.mark.parametrize("mask", [0.0, 0.4])
def test_lone_walkers_send_their_own_rows(n, depth, mask):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(n + depth, n_expand=2 * n + 40, fanout=(1, 90 if n < 300 else 9), max_depth=70, n_roots=n, mask_frac=mask)
    ref = R.RefTree.from_soa(soa)
    f = omk.Forest.from_soa(soa)
    b = omk.Batch(f, n, depth)
    b.set_roots(roots[:n])
    rng = np.random.default_rng(n)
    for step in range(6):
        rpaths, rlen, rleaf, _ = ref.select_batch(roots[:n], R.make_params(c_puct=1.4, virtual_loss=3, max_depth=depth))
        values = (rng.integers(-64, 65, n) / 64.0).astype(np.float32)
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        b.set_values(values)
        if step == 3:
            ref.backup_batch(rpaths, rlen, values, 3)
            b.backup(3)
        for _ in range(0 if step == 4 else 2):
            paths, plen, leaf, actions = b.read()
            assert (paths == rpaths).all() and (plen == rlen).all() and (leaf == rleaf).all()
            assert (actions == ref.gather_actions(rpaths, rlen)).all()
        if step != 3:
            ref.backup_batch(rpaths, rlen, values, 3)
            b.backup(3)
        got = f.download()
        assert (got["N"] == ref.N).all() and (got["W"] == ref.W).all() and (got["VL"] == ref.VL).all()


# two batches on one forest: what one of them has staged, after a wrap of the staging, is still on its way when the
# other one reads rows its walkers sent before and stages again
def test_values_staged_behind_a_lone_selection_arrive_whole():
    import omoknuni_small_amd as omk
    soa, roots = random_tree(81, n_expand=900, fanout=(1, 9), max_depth=6, n_roots=300)
    ref = R.RefTree.from_soa(soa)
    f = omk.Forest.from_soa(soa)
    rng = np.random.default_rng(81)
    many = 600_000  # 2.4 of the 4 MB: the second time they do not fit behind the first
    params = omk.SelectParams(c_puct=1.4, virtual_loss=3)
    lone, other = omk.Batch(f, 256, 6), omk.Batch(f, many, 6)
    lone.set_roots(roots[:256])
    other.set_roots(roots[256:])
    first, second, own = ((rng.integers(-64, 65, n) / 64.0).astype(np.float32) for n in (many, many, 256))
    for step in range(4):
        rlone = ref.select_batch(roots[:256], R.make_params(c_puct=1.4, virtual_loss=3, max_depth=6))
        rother = ref.select_batch(roots[256:], R.make_params(c_puct=1.4, virtual_loss=3, max_depth=6))
        other.select(params)
        other.set_values(first)
        lone.select(params)
        other.set_values(second)
        paths, plen, leaf, _ = lone.read()
        lone.set_values(own)
        other.backup(3)
        lone.backup(3)
        assert (paths == rlone[0]).all() and (plen == rlone[1]).all() and (leaf == rlone[2]).all()
        ref.backup_batch(rother[0], rother[1], second[:44], 3)
        ref.backup_batch(rlone[0], rlone[1], own, 3)
        got = f.download()
        assert (got["N"] == ref.N).all() and (got["VL"] == ref.VL).all()
        err = np.abs(got["W"].astype(np.float64) - ref.W) / np.maximum(np.abs(ref.W), 1.0)
        assert err.max() <= 1e-5, step  # (the trees' own sums are no multiples of 1/64)
        ref.W[:] = got["W"]
        first, second = second, first


# what a batch needs to be read and expanded it has from its creation: the device's mappings stay as they are
# (the largest takes more than the 16 MB of pinned memory a batch has for it: it crosses in pieces)
@pytest.mark.parametrize("n,depth", [(1, 5), (40, 12), (3000, 30), (90_000, 30)])
def test_the_first_read_and_expansion_of_a_batch_allocate_nothing(n, depth):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(3, n_expand=300, fanout=(1, 5), max_depth=10, n_roots=40)
    begin = np.arange(n + 1, dtype=np.int32)
    moves = np.zeros(n, np.int32)
    f = omk.Forest.from_soa(soa, capacity=len(soa["N"]) + 8 * n)
    same = []
    for _ in range(4):  # (the first batch brings in the kernels, and the runtime may map something of its own now and then)
        b = omk.Batch(f, n, depth)
        b.set_roots(roots[np.arange(n) % 40])
        before = mapped()
        for _ in range(2):
            b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
            b.read()
            b.expand(begin, moves)
            b.revert_vl(3)
        same.append(mapped() == before)
        b.close()
    assert any(same[1:])


# a gather of more than 16 MB crosses in pieces of half of that: one traversal short of it, one beyond, pieces that
# end with the last traversal and that do not, the deepest paths there are
@pytest.mark.parametrize("n,depth", [(64_527, 30), (64_528, 30), (3 * 32_256, 30), (3 * 32_256 + 1, 30), (577, 4096)])
def test_gathers_in_pieces(n, depth):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(9, n_expand=900, fanout=(1, 5), max_depth=40, n_roots=300)
    ref = R.RefTree.from_soa(soa)
    troots = roots[np.arange(n) % 300]
    rpaths, rlen, rleaf, _ = ref.select_batch(troots, R.make_params(c_puct=1.4, virtual_loss=3, max_depth=depth))
    f = omk.Forest.from_soa(soa, capacity=ref.n + 3 * n)
    b = omk.Batch(f, n, depth)
    b.set_roots(troots)
    b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
    paths, plen, leaf, actions = b.read()
    assert (paths == rpaths).all() and (plen == rlen).all() and (leaf == rleaf).all()
    assert (actions == ref.gather_actions(rpaths, rlen)).all()
    # and what an expansion takes from it
    begin = np.arange(n + 1, dtype=np.int32) * 3
    moves = np.tile(np.int32([4, 1, 7]), n)
    assert (b.expand(begin, moves) == ref.expand_batch(rleaf, begin, moves)).all()


# an expansion that has to gather the leaves itself, of so many traversals that they cross in pieces
def test_an_expansion_of_more_than_a_million_traversals():
    import omoknuni_small_amd as omk
    n = (1 << 20) + 77
    zeros = np.zeros(n, np.int32)
    soa = dict(N=zeros, W=np.zeros(n, np.float32), P=np.ones(n, np.float32), VL=zeros, child_begin=zeros,
               child_count=zeros, action=zeros - 1)
    f = omk.Forest.from_soa(soa, capacity=2 * n)
    b = omk.Batch(f, n, 3)
    b.set_roots(np.arange(n, dtype=np.int32))
    b.select(omk.SelectParams(c_puct=1.4, virtual_loss=1))
    counts = (np.arange(n) % 3 > 0).astype(np.int32)  # every third position is over
    begin = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    first = b.expand(begin, np.arange(begin[-1], dtype=np.int32))
    assert (first == np.where(counts > 0, n + begin[:-1], -1)).all()
    sx = f.download_structure()
    assert (sx["child_begin"][:n][counts > 0] == first[counts > 0]).all() and (sx["child_count"][:n] == counts).all()
    assert (sx["action"][n:] == np.arange(begin[-1])).all()


# roots, values and keys beyond the 4 MB of staging cross in pieces, and take no pinned memory beside it
@pytest.mark.parametrize("doubled", [0, 70_000])
def test_large_batches_are_handed_over_in_pieces(doubled):
    import omoknuni_small_amd as omk
    n_roots, n = 400_000, 400_000 + doubled  # the first roots have two traversals each
    rng = np.random.default_rng(doubled)
    nodes = 3 * n_roots
    soa = dict(N=rng.integers(1, 9, nodes).astype(np.int32), W=rng.integers(-4, 5, nodes).astype(np.float32),
               P=rng.random(nodes).astype(np.float32), VL=np.zeros(nodes, np.int32), child_begin=np.zeros(nodes, np.int32),
               child_count=np.zeros(nodes, np.int32), action=np.tile(np.arange(3, dtype=np.int32), n_roots),
               hash=np.zeros(nodes, np.uint64))
    soa["child_begin"][:n_roots], soa["child_count"][:n_roots] = n_roots + 2 * np.arange(n_roots), 2
    troots = rng.permutation(np.arange(n, dtype=np.int32) % n_roots)
    ref = R.RefTree.from_soa(soa)
    rpaths, rlen, rleaf, _ = ref.select_batch(troots, R.make_params(c_puct=1.4, virtual_loss=3, max_depth=2))
    keys = rng.permutation(np.arange(1, nodes + 1, dtype=np.uint64))
    values = (rng.integers(-64, 65, n) / 64.0).astype(np.float32)
    same = []
    for last in (False, False, False, True):  # (as above)
        f = omk.Forest.from_soa(soa)
        b = omk.Batch(f, n, 2)
        before = mapped()
        b.set_roots(troots)
        b.set_values(values)
        f.set_keys(np.arange(nodes, dtype=np.int32), keys)
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        paths, plen, leaf, _ = b.read()
        same.append(mapped() == before)
        assert (paths == rpaths).all() and (plen == rlen).all() and (leaf == rleaf).all()
        if not last:
            b.close()
            f.close()
    assert any(same[1:])
    table = omk.TranspositionTable(f, 21)
    table.insert(keys[::3], np.arange(nodes, dtype=np.int32)[::3])
    assert (table.probe_leaves(b) == np.where(leaf % 3 == 0, leaf, -1)).all()
    b.backup(3)
    ref.backup_batch(rpaths, rlen, values, 3)
    got = f.download()
    assert (got["N"] == ref.N).all() and (got["VL"] == ref.VL).all() and (got["W"] == ref.W).all()


# offers of more than 4 MB: pieces of whole leaves, with a legal mask (whose words pieces share) and without
@pytest.mark.parametrize("mask", [0.0, 0.3])
@pytest.mark.parametrize("moves,n", [(1000, 700), (33, 16_500)])
def test_an_expansion_in_pieces(moves, n, mask):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(12, n_expand=300, fanout=(1, 3), max_depth=2, n_roots=n, mask_frac=mask, vl_frac=0.0)
    ref = R.RefTree.from_soa(soa)
    f = omk.Forest.from_soa(soa, capacity=ref.n + n * moves)
    b = omk.Batch(f, n, 4)
    b.set_roots(roots[:n])
    rleaf = ref.select_batch(roots[:n], R.make_params(c_puct=1.4, virtual_loss=3, max_depth=4))[2]
    b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
    rng = np.random.default_rng(moves)
    counts = rng.integers(moves - 3, moves + 1, n)
    begin = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    mv = rng.integers(0, 1200, begin[-1]).astype(np.int32)
    policy = rng.random(begin[-1]).astype(np.float32)  # one value a child
    got = b.expand_ex(begin, mv, begin, policy, 2000)
    assert (got == ref.expand_batch(rleaf, begin, mv, policy=policy, action_space=2000, policy_begin=begin)).all()
    st, sx = f.download(), f.download_structure()
    assert (st["N"] == ref.N).all() and st["P"].tobytes() == ref.P.tobytes() and (st["VL"] == ref.VL).all()
    assert (sx["child_begin"] == ref.child_begin).all() and (sx["child_count"] == ref.child_count).all()
    assert (sx["action"] == ref.action).all()
    # the new children take part in the next selection as the checker has them
    rpaths, rlen, _, _ = ref.select_batch(roots[:n], R.make_params(c_puct=1.4, virtual_loss=3, max_depth=4))
    b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
    paths, plen, _, _ = b.read()
    assert (paths == rpaths).all() and (plen == rlen).all()


# what an expansion takes from rows that the walkers have sent: the leaves, whether they have children already (the
# depth bound) and their visits (the widening); sent by blocks up to 256 traversals, by wavefronts up to 128
@pytest.mark.parametrize("n", [1, 3, 128, 129, 256, 257])
@pytest.mark.parametrize("fanout,mask", [((1, 6), 0.0), ((1, 6), 0.4), ((60, 90), 0.4)])
def test_expansion_after_lone_walkers_have_sent_their_rows(n, fanout, mask):
    import omoknuni_small_amd as omk
    soa, roots = random_tree(n + 17, n_expand=n + 30, fanout=fanout, max_depth=4, n_roots=n, mask_frac=mask, n_max=400, vl_frac=0.0)
    depth = 2 if fanout[1] < 64 else 1  # so that some leaves have children
    ref = R.RefTree.from_soa(soa)
    moves, A = 60, 200
    f = omk.Forest.from_soa(soa, capacity=ref.n + 3 * n * moves)
    b = omk.Batch(f, n, depth)
    b.set_roots(roots[:n])
    rng = np.random.default_rng(n)
    kept = widened = 0
    for step in range(3):
        rpaths, rlen, rleaf, _ = ref.select_batch(roots[:n], R.make_params(c_puct=1.4, virtual_loss=3, max_depth=depth))
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        paths, plen, leaf, actions = b.read()
        assert (paths == rpaths).all() and (plen == rlen).all() and (leaf == rleaf).all()
        assert (actions == ref.gather_actions(rpaths, rlen)).all()
        kept += int((ref.child_count[rleaf] > 0).sum())
        begin = (np.arange(n + 1) * moves).astype(np.int32)
        mv = np.concatenate([rng.permutation(A)[:moves] for _ in range(n)]).astype(np.int32)
        policy = rng.random((n, A)).astype(np.float32)
        at = ref.n
        want = ref.expand_batch(rleaf, begin, mv, policy=policy, action_space=A, widening=(2.0, 0.5))
        widened += int((ref.child_count[rleaf[want >= at]] > 8).sum())
        got = b.expand_ex(begin, mv, (np.arange(n + 1) * A).astype(np.int32), policy, A, widening=(2.0, 0.5))
        assert (got == want).all()
        values = (rng.integers(-64, 65, n) / 64.0).astype(np.float32)
        ref.backup_batch(rpaths, rlen, values, 3)
        b.set_values(values)
        b.backup(3)
        st, sx = f.download(), f.download_structure()
        ref.W[:] = st["W"]
        assert (st["N"] == ref.N).all() and st["P"].tobytes() == ref.P.tobytes() and (st["VL"] == ref.VL).all()
        assert (sx["child_begin"] == ref.child_begin).all() and (sx["child_count"] == ref.child_count).all()
    assert n < 100 or (kept > 0 and widened > 0)
