"""GPU parity of the node whose visitors split between children, settled by the helpers of its block at once, at the edges
of what it takes: visitors (few, what one batch of entries holds, the most before a node is cut into slices), fan-out
classes, and keys that pile up (plateaus, exactly tied children, one child that takes nearly all)."""
import numpy as np
import pytest

from test_gpu_scheduler import layered_forest, select_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("visitors", [66, 193, 700, 1475, 1535, 1536])
@pytest.mark.parametrize("fan,rave,plateau", [(3, False, False), (64, False, False), (65, True, True), (256, True, False),
                                              (384, True, True), (385, False, False), (1000, True, True)])
def test_crowds_and_fan_outs(visitors, fan, rave, plateau):
    soa, roots = layered_forest(fan + visitors, [fan, 30, 4], rave=rave, plateau=plateau)
    st = select_both(soa, np.zeros(visitors, np.int32), 4, rave=rave)
    assert st["merged_nodes"] + st["sliced_nodes"] >= 1, st
    assert st["replayed_nodes"] == 0, st


@pytest.mark.parametrize("fan", [40, 300, 600])
@pytest.mark.parametrize("kind", ["tied", "fresh", "dominated"])
def test_keys_that_pile_up(fan, kind):
    """All children exactly alike (visited or not): every key occurs in every child; one that outweighs the rest together."""
    soa, roots = layered_forest(fan, [fan, 20])
    kids = slice(1, 1 + fan)
    soa["N"][kids], soa["W"][kids], soa["P"][kids] = (0, 0.0, 1.0 / fan) if kind == "fresh" else (50, 5.0, 1.0 / fan)
    if kind == "dominated":
        soa["N"][7], soa["W"][7], soa["P"][7] = 100_000, 20_000.0, 0.5
    for visitors in (100, 1500):
        st = select_both(soa, np.zeros(visitors, np.int32), 3, steps=3)
        assert st["merged_nodes"] >= 1, st


@pytest.mark.parametrize("visitors", [70, 256, 512, 1475, 1535])
@pytest.mark.parametrize("fan", [24, 240, 362])
def test_blends_that_stop_moving(visitors, fan):
    """RAVE blends of much visited children: after a few visitors the sum rounds to one score, and the closed form, which
    knows of no rounding, sees none of the entries that lie on it."""
    rng = np.random.default_rng(fan)
    n = fan + 1
    N = np.r_[900_000, rng.integers(0, 400, fan)].astype(np.int32)
    W = (rng.uniform(-0.5, 0.5, n) * N).astype(np.float32)
    P = np.full(n, 1e-4, np.float32)
    rN = np.full(n, 1000, np.int32)
    rW = rng.integers(-500, 500, n).astype(np.float32)
    a, b, c = 1 + rng.choice(fan, 3, replace=False)
    N[a], W[a], P[a], rW[a] = 889_482, 888_997.0, 0.0068, -800.0
    N[b], W[b], P[b], rW[b] = 892_192, 891_680.75, 0.00035, 990.0
    N[c], W[c], P[c], rW[c] = 650_000, 649_600.0, 0.0004, 992.0
    first = np.r_[1, np.zeros(fan)].astype(np.int32)
    soa = dict(N=N, W=W, P=P, VL=np.zeros(n, np.int32), child_begin=first, child_count=first * fan,
               action=np.r_[-1, np.arange(fan)].astype(np.int32), rN=rN, rW=rW)
    st = select_both(soa, np.zeros(visitors, np.int32), 3, rave=True, steps=1)
    assert st["merged_nodes"] == st["group_nodes"] == 1 and st["replayed_nodes"] == 0, st
