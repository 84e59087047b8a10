"""GPU parity of the selection of batches whose roots have at most 64 visitors each (a block a root) at the edges of what
it takes: visitors of a root, fan-out classes, roots with one visitor among the others, depth bounds, values without a
real score; and of the rows the blocks send to the host themselves."""
import numpy as np
import pytest

from helpers import random_tree, star
from oracle import ref_cpu as R
from test_gpu_scheduler import layered_forest

pytestmark = pytest.mark.gpu


def both(soa, troots, D, vl=3, rave=False, pw=False, steps=4, count=False):
    """Selections and backups on the device and by the checker; from the second on the rows come from the blocks.  With
    `count` the work counters are on, and their sums are returned."""
    import omoknuni_small_amd as omk
    ref = R.RefTree.from_soa(soa)
    rp = R.make_params(c_puct=1.4, virtual_loss=vl, use_rave=rave, rave_k=1000.0, pw=pw, max_depth=D)
    f = omk.Forest.from_soa(soa)
    b = omk.Batch(f, len(troots), D)
    b.set_roots(troots)
    sp = omk.SelectParams(c_puct=1.4, virtual_loss=vl, use_rave=rave, rave_k=1000.0, pw=pw)
    rng = np.random.default_rng(len(troots))
    b.enable_stats(count)
    total = {}
    for step in range(steps):
        rpaths, rlen, rleaf, _ = ref.select_batch(troots, rp, near_ties=False)
        b.select(sp)
        paths, plen, leaf, acts = b.read()
        assert (paths == rpaths).all() and (plen == rlen).all() and (leaf == rleaf).all(), step
        assert (acts == ref.gather_actions(rpaths, rlen)).all(), step
        if count:
            total = {k: v + total.get(k, 0) for k, v in b.stats().items()}
        assert b.truncated() == int(((ref.child_count[rleaf] > 0) & (rlen == D + 1)).sum()), step
        values = (rng.integers(-64, 65, len(troots)) / 64.0).astype(np.float32)
        was, visits = ref.W.astype(np.float64), ref.N.copy()
        ref.backup_batch(rpaths, rlen, values, vl)
        b.set_values(values)
        b.backup(vl)
        got = f.download()
        assert (got["N"] == ref.N).all() and (got["VL"] == ref.VL).all(), step
        # k values of at most 1 added to W in two orders: every partial sum is at most |W| + k and rounds by 2^-24 of it
        k, finite = ref.N - visits, np.isfinite(was)
        bound = 2.0 ** -23 * k[finite] * (np.abs(was[finite]) + k[finite])
        assert (np.abs(got["W"][finite].astype(np.float64) - ref.W[finite]) <= bound).all(), step
        assert np.array_equal(got["W"][~finite], ref.W[~finite], equal_nan=True), step
        ref.W[:] = got["W"]
    return total


@pytest.mark.parametrize("visitors", [2, 3, 17, 63, 64, 65])
@pytest.mark.parametrize("fan,rave", [(2, False), (64, True), (65, False), (256, False), (257, True), (384, True),
                                      (385, False)])
def test_crowds_and_fan_outs(visitors, fan, rave):
    soa, roots = layered_forest(3 + fan + visitors, [fan, 40, 5], n_trees=3, rave=rave)
    both(soa, np.repeat(roots, visitors).astype(np.int32), 6, rave=rave)


@pytest.mark.parametrize("visitors", [8, 33, 64])
@pytest.mark.parametrize("fan,rave", [(3, False), (64, True), (256, False), (384, True)])
@pytest.mark.parametrize("rising", [False, True])
def test_contested_nodes_are_merged_unless_scores_rise(visitors, fan, rave, rising):
    """What spreads is merged and nothing is replayed; children whose scores rise with virtual loss (a value sum below minus
    the visit count) are not in order, and their node is replayed: with the same paths."""
    soa, roots = layered_forest(fan + visitors, [fan, 20, 4], n_trees=3, rave=rave)
    if rising:
        soa["N"] = np.maximum(soa["N"], 1)
        soa["W"] = (-np.random.default_rng(fan).uniform(1.5, 2.5, len(soa["N"])) * soa["N"]).astype(np.float32)
        soa["P"][:] = 0.0
        if rave:  # (and the blend is no better)
            soa["rN"] = np.maximum(soa["rN"], 1)
            soa["rW"] = (-5.0 * soa["rN"]).astype(np.float32)
    st = both(soa, np.repeat(roots, visitors).astype(np.int32), 6, rave=rave, count=True)
    if rising:
        assert st["replayed_nodes"] >= 1, st
    else:
        assert st["merged_by_blocks"] >= 1 and st["replayed_nodes"] == 0, st
    assert st["settled_one_by_one"] >= 2 * st["replayed_nodes"], st


@pytest.mark.parametrize("rave", [False, True])
@pytest.mark.parametrize("widest,mask", [(12, 0.0), (150, 0.4), (380, 0.3)])
@pytest.mark.parametrize("D", [1, 7, 63, 64])
def test_roots_of_all_sizes_in_one_batch(widest, mask, D, rave):
    """Roots with 1 to 64 visitors side by side (the single ones in blocks of their own), ties, unvisited children, virtual
    loss from before; rows only where the bound is below 64."""
    soa, roots = random_tree(D + widest, n_expand=120, fanout=(2, widest), max_depth=9, n_roots=40, mask_frac=mask, rave=rave,
                             vl_frac=0.1, tie_frac=0.1, n_max=200)
    rng = np.random.default_rng(D)
    sizes = np.concatenate([np.ones(19, np.int64), rng.integers(2, 65, 21)])
    both(soa, rng.permutation(np.repeat(roots, sizes)).astype(np.int32), D, rave=rave)


@pytest.mark.parametrize("crowds", [[64, 2, 33], [2], [65]])
@pytest.mark.parametrize("widest,mask,rave,n_expand", [(12, 0.0, False, 5000), (150, 0.4, True, 1500)])
@pytest.mark.parametrize("alternating", [False, True])
def test_few_crowded_roots_among_thousands_of_lone_ones(crowds, widest, mask, rave, n_expand, alternating):
    """Up to 64 visitors a root the lone ones are walked by blocks of 16 beside the crowds' own; from 65 on by the walkers
    of the persistent launch."""
    lone = 2503
    soa, roots = random_tree(n_expand, n_expand=n_expand, fanout=(2, widest), max_depth=6, n_roots=len(crowds) + lone,
                             mask_frac=mask, rave=rave, tie_frac=0.1, n_max=200)
    troots = np.repeat(roots, crowds + [1] * lone).astype(np.int32)
    both(soa, np.random.default_rng(lone).permutation(troots) if alternating else troots, 9, rave=rave, steps=2)


@pytest.mark.parametrize("visitors", [1, 2, 3, 4, 13, 64])
@pytest.mark.parametrize("fan,rave", [(3, False), (64, True), (65, False), (225, False), (384, True)])
def test_scores_closer_than_their_bounds(visitors, fan, rave):
    """Scores that differ by nothing or by a few units in the last place, which the bounds (2^-18 wide) cannot tell apart,
    among children with and without visits: crowds, and lone visitors beside them."""
    soa, roots = layered_forest(fan + 7 * visitors, [fan, 30, 5], n_trees=4, rave=rave)
    rng = np.random.default_rng(fan + visitors)
    n = len(soa["N"])
    near = rng.random(n) < 0.8
    near[roots] = False
    soa["N"] = np.where(near, np.where(rng.random(n) < 0.3, 0, 200), soa["N"]).astype(np.int32)
    soa["W"] = np.where(near, soa["N"] / 4.0, soa["W"]).astype(np.float32)
    p = np.float32(1.0 / fan)
    steps = rng.integers(-3, 4, n)
    soa["P"] = np.where(near, p * (np.float32(1) + steps.astype(np.float32) * np.float32(2.0 ** -23)), soa["P"]).astype(np.float32)
    if rave:
        soa["rN"] = np.where(near, 0, soa["rN"]).astype(np.int32)
        soa["rW"] = np.where(near, 0.0, soa["rW"]).astype(np.float32)
    both(soa, np.repeat(roots, [visitors, 1, max(1, visitors - 1), visitors]).astype(np.int32), 6, rave=rave)


@pytest.mark.parametrize("kind", ["nan prior", "nan sum", "-inf sum", "inf sum of the unvisited", "no virtual loss", "all equal",
                                  "next to nothing"])
@pytest.mark.parametrize("rave", [False, True])
def test_scores_that_are_not_real_and_ties(kind, rave):
    soa, roots = random_tree(11, n_expand=60, fanout=(2, 130), max_depth=6, n_roots=6, rave=rave, n_max=30)
    rng = np.random.default_rng(5)
    some = rng.random(len(soa["N"])) < 0.3
    some[roots] = False
    if kind == "nan prior":
        soa["P"][some] = np.nan
    elif kind == "nan sum":
        soa["W"][some] = np.nan
    elif kind == "-inf sum":
        soa["W"][some] = -np.inf
    elif kind == "inf sum of the unvisited":
        soa["W"][some & (soa["N"] == 0)] = np.inf
    elif kind == "all equal":
        soa["N"][:], soa["W"][:], soa["P"][:] = 1, 0.5, 0.25
    elif kind == "next to nothing":  # quotients that underflow, which the bounds cannot tell apart
        soa["W"][:], soa["P"] = 0.0, (rng.integers(0, 64, len(some)) * 2.0 ** -149).astype(np.float32)
        if rave:
            soa["rW"][:] = 0.0
    both(soa, np.repeat(roots, 20).astype(np.int32), 8, vl=0 if kind == "no virtual loss" else 2, rave=rave, steps=1)


@pytest.mark.parametrize("visitors", [1, 2, 3, 4, 20, 64])
@pytest.mark.parametrize("fan", [2, 5, 63, 70])
def test_unvisited_children_whose_sums_are_not_finite(visitors, fan):
    """A child nobody has visited is scored without its sum, and with it from its first visitor on: where no sum is finite
    the first scan has a real score for the first `fan` visitors only, and the others take the least visited child, although
    the RAVE blends of the second scan stay real."""
    for bad in (np.nan, np.inf, -np.inf):
        soa = star(200, [[0, bad, 7.1e-8 * (1 + i / 1000), 0, 10, 5] for i in range(fan)], rave=True)
        both(soa, np.zeros(visitors, np.int32), 2, rave=True, steps=1)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("field", ["P", "W"])
@pytest.mark.parametrize("fan,rave", [(9, False), (225, False), (362, True)])
def test_empty_slots_whose_values_are_not_finite(fan, rave, field, value):
    """What stands in a slot without a legal move is looked at by nobody: crowds and lone visitors are settled as if it were
    zero there, and no more of them one after the other."""
    soa, roots = layered_forest(fan + rave, [fan, 20, 4], n_trees=3, rave=rave)
    n = len(soa["N"])
    legal = np.random.default_rng(fan).random((n + 31) // 32 * 32) < 0.6
    legal[roots] = True
    legal[soa["child_begin"][soa["child_count"] > 0]] = True
    soa["legal"] = np.packbits(legal.reshape(-1, 32), axis=1, bitorder="little").view("<u4").reshape(-1).copy()
    sums = []
    for v in (0.0, value):
        soa[field] = np.where(legal[:n], soa[field], np.float32(v)).astype(np.float32)
        st = both(soa, np.repeat(roots, [64, 1, 9]).astype(np.int32), 6, rave=rave, count=True)
        sums.append({k: c for k, c in st.items() if not k.startswith("t_")})
    assert sums[0] == sums[1] and sums[1]["settled_one_by_one"] == 0, sums


@pytest.mark.parametrize("visitors", [2, 3])
@pytest.mark.parametrize("fan", [3, 64, 65, 130, 380])
def test_few_visitors_look_at_the_listed_children_only(fan, visitors):
    """Two or three visitors who split between the first and the last child (from 65 children on of one lane, or of two); the
    others are ruled out, and that one of them would do better with every visit is no reason to replay the node."""
    kids = [[100, 90.0, 0.3, 0, 0, 0.0]] + [[0, 10.0, 0.0, 0, 100, 1.0]] * (fan - 2) + [[100, 90.0, 0.3, 0, 0, 0.0]]
    for last in (fan - 1, 64):  # the same lane and the next one, or the last
        if last < fan:
            kids[fan - 1], kids[last] = kids[last], kids[fan - 1]
            st = both(star(400, kids, rave=True), np.zeros(visitors, np.int32), 2, rave=True, steps=1, count=True)
            assert st["replayed_nodes"] == 0 and st["settled_one_by_one"] == 0, st


def test_widening_at_the_selection():
    soa, roots = random_tree(21, n_expand=80, fanout=(2, 200), max_depth=7, n_roots=9, sort_prior=True, n_max=400)
    both(soa, np.repeat(roots, [1, 2, 5, 9, 16, 33, 48, 63, 64]).astype(np.int32), 8, pw=True)


@pytest.mark.parametrize("sizes", [[64], [2, 64, 17, 1, 1, 1, 40], [1] * 50, [65], [700, 3, 1, 1], [5000, 80, 1]])
@pytest.mark.parametrize("fan,rave", [(48, False), (300, True)])
def test_work_counters(sizes, fan, rave):
    """The counters against the paths: a node with several visitors that go on from it is one processed node, a lone
    visitor's step is one, and every merge has been made by a team or by a block."""
    import omoknuni_small_amd as omk
    soa, roots = layered_forest(fan, [fan, 8, 4], n_trees=len(sizes), rave=rave)
    troots = np.repeat(roots, sizes).astype(np.int32)
    b = omk.Batch(omk.Forest.from_soa(soa), len(troots), 6)
    b.set_roots(troots)
    b.enable_stats()
    for _ in range(3):  # (the rows of the last two come from the blocks)
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3, use_rave=rave, rave_k=1000.0))
        paths, plen, _, _ = b.read()
        st = b.stats()
        went_on = paths[:, :-1][np.arange(paths.shape[1] - 1)[None, :] < plen[:, None] - 1]
        visitors = np.bincount(went_on)
        assert st["group_nodes"] == (visitors > 1).sum()
        assert st["settled_by_water_level"] + st["settled_one_by_one"] == visitors[visitors > 1].sum()
        assert st["single_visitor_steps"] == (visitors == 1).sum()
        assert st["merged_by_teams"] + st["merged_by_blocks"] == st["merged_nodes"]
        assert (st["merged_by_blocks"] > 0) == (1 < max(sizes) <= 64) and (st["merged_by_teams"] > 0) == (max(sizes) > 64)
        b.backup(3)


def test_time_stamps():
    """When the first block started and the last one left: around all work of the timeline, of this selection and not of an
    earlier one, whether the rows come from the blocks or not; with the counters and the timeline off only the persistent
    launch keeps them."""
    import omoknuni_small_amd as omk
    soa, roots = random_tree(77, n_expand=900, fanout=(2, 150), max_depth=9, n_roots=300, n_max=200)
    f = omk.Forest.from_soa(soa)
    few = np.repeat(roots, np.r_[64, np.full(149, 6), np.ones(150, np.int64)]).astype(np.int32)
    many = np.repeat(roots[:3], 70).astype(np.int32)
    b = omk.Batch(f, len(few), 12)
    before = None
    for troots, trace, read in [(few, True, False), (few, True, True), (few, True, True), (many, False, True), (few, False, True),
                                (roots.astype(np.int32), True, True), (many, True, True), (few, True, True)]:
        b.set_roots(troots)
        b.enable_trace(trace)
        b.select(omk.SelectParams(c_puct=1.4, virtual_loss=3))
        if read:
            b.read()
        st = b.stats()
        b.revert_vl(3)
        first, last = st["t_first_block"], max(st["t_last_team"], st["t_last_walker"])
        if len(troots) == 300 or troots is few and not trace:
            assert first == last == 0
            continue
        assert (st["t_last_walker"] != 0) == (troots is many)
        assert before is None or (first - before) % (1 << 31) < 1 << 30
        assert 0 < (last - first) % (1 << 31) < 10_000_000  # (a tenth of a second)
        if trace:  # (the block numbered first need not be the first to start: 10 us)
            tr = b.debug_trace()
            assert len(tr) > 0 and ((tr[:, 0] - first + 1000) % (1 << 31) < 1 << 30).all()
            assert ((last - tr[:, 1]) % (1 << 31) < 1 << 30).all()
        before = last


@pytest.mark.parametrize("kind", ["nan sum", "no score at all", "all equal"])
@pytest.mark.parametrize("widest,rave", [(60, False), (250, True), (380, False), (380, True)])
def test_lone_visitors_of_masked_trees(widest, rave, kind):
    """One visitor a root, a block a visitor with a wavefront for every 64 children: ties across wavefronts, wavefronts
    without a real score, nodes without one (the least visited child is taken)."""
    soa, roots = random_tree(31, n_expand=90, fanout=(2, widest), max_depth=6, n_roots=30, mask_frac=0.3, rave=rave, n_max=30)
    some = np.random.default_rng(6).random(len(soa["N"])) < 0.5
    some[roots] = False
    if kind == "all equal":
        soa["N"][:], soa["W"][:], soa["P"][:] = 1, 0.5, 0.25
    else:
        soa["P" if kind == "no score at all" else "W"][some if kind == "nan sum" else slice(None)] = np.nan
    both(soa, np.array(roots, np.int32), 8, vl=2, rave=rave, steps=1)
