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
