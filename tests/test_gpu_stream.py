"""Large launches against small ones: a level whose first-stage fluxes are
stored past the caches and whose transverse and final fluxes are joined, and
the same level in slabs too thin for either, bit for bit."""
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


@pytest.mark.parametrize("n,bc", [((80, 80, 80), 1), ((129, 63, 62), 0), ((31, 33, 490), 1)])
def test_whole_level_matches_thin_slabs(n, bc):
    hi = tuple(v / 16.0 for v in n)
    cfg = small_cfg(n=16, bc=bc)
    S = mixed_flow(n, seed=sum(n))
    out = []
    for slab in (0, 7):
        L = mc.Level(n, configs.grid_boxes(n, 512), cfg["prob_lo"], hi, bc, mc.MODE_FUSED)
        L.set_fused_slab(slab)
        L.set_state(S)
        L.run(3)
        out.append((L.state(), L.dt, L.time))
        L.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]
