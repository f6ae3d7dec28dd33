"""The ring of planes that holds an engine's primitives in slabs: large levels
in slabs, shallow and deep, with a last slab of fewer planes, equal the
whole-level engine bit for bit."""
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


@pytest.mark.parametrize("n,bc,slab,tflux", [((127, 126, 126), 0, 31, None), ((130, 128, 121), 1, 17, None),
                                             ((420, 360, 14), 0, 1, None), ((420, 360, 14), 1, 1, (8, 32, 64)),
                                             ((410, 408, 13), 0, 4, (8, 32, 64)), ((410, 408, 12), 1, 3, (4, 64, 64))])
def test_large_level_in_slabs_matches_whole_level(n, bc, slab, tflux):
    """With slabs shallower than the z-bricks of the first-stage fluxes too."""
    hi = tuple(v / 16.0 for v in n)
    cfg = small_cfg(n=16, bc=bc)
    S = mixed_flow(n, seed=sum(n) + bc)
    out = []
    for planes in (0, slab):
        L = mc.Level(n, configs.grid_boxes(n, 512), cfg["prob_lo"], hi, bc, mc.MODE_FUSED)
        L.set_fused_slab(planes)
        L.set_state(S)
        if tflux:
            L.set_tiling(L.STAGES.index("tflux"), *tflux)
        L.run(1, use_graph=False)
        L.run(2, use_graph=True)
        out.append((L.state(), L.dt, L.time))
        L.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]
