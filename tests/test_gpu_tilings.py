"""The brick an engine starts with in the stages that solve the EOS cell by
cell: narrower rows where rows of 64 stick out of a large domain, and the same
bits as with rows of 64."""
import numpy as np
import pytest

import minicastro as mc
from minicastro import configs
from helpers import small_cfg, table_bin
from test_gpu_species import mixed_flow

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu_table():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())


@pytest.mark.parametrize("n,brick", [((48, 48, 48), (16, 4, 2)), ((96, 36, 30), (32, 2, 2)), ((64, 40, 41), (64, 4, 1)),
                                     ((40, 40, 40), (64, 4, 1))])
def test_brick_of_the_cell_stages(n, brick):
    hi = tuple(v / 16.0 for v in n)
    cfg = small_cfg(n=16, bc=0)
    states = []
    for wide in (False, True):
        L = mc.Level(n, configs.grid_boxes(n, 512), cfg["prob_lo"], hi, 0, mc.MODE_FUSED)
        L.set_state(mixed_flow(n, seed=7))
        L.coarse_step()
        for st in ("est", "prim", "update"):
            if not wide:
                assert L.get_tiling(L.STAGES.index(st)) == brick
            L.set_tiling(L.STAGES.index(st), *((64, 4, 1) if wide else brick))
        L.run(2)
        states.append((L.state(), L.dt, L.time))
        L.close()
    np.testing.assert_array_equal(states[0][0], states[1][0])
    assert states[0][1:] == states[1][1:]
