"""The transverse and final fluxes joined in one launch (K_transfinal), which
levels and slabs of 200,000 cells and more take: bit for bit against the
oracle, at sizes where its tiles and chunks leave remainders, for both
boundaries, in slabs of which the last is too small for it, and with the
other stages' variants."""
import numpy as np
import pytest

import minicastro as mc
from minicastro import configs
from helpers import oracle_level, small_cfg, table_bin
from test_gpu_species import mixed_flow

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu_table():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())


# n_cell, bc, planes of a slab (0: whole), stage variant
CASES = [((57, 61, 59), 0, 0, 0), ((29, 15, 461), 1, 0, 5), ((4, 225, 224), 0, 0, 4), ((120, 70, 30), 1, 24, 1)]


@pytest.mark.parametrize("n,bc,slab,variant", CASES)
def test_joined_fluxes_match_oracle(n, bc, slab, variant):
    hi = tuple(v / 16.0 for v in n)
    cfg = small_cfg(n=16, bc=bc)
    cfg.update(n_cell=n, prob_hi=hi, boxes=configs.grid_boxes(n, 512))
    S = mixed_flow(n, seed=sum(n) + bc)
    O = oracle_level(cfg, nthreads=8)
    O.set_state(S)
    G = mc.Level(n, cfg["boxes"], cfg["prob_lo"], hi, bc, mc.MODE_FUSED)
    G.set_fused_slab(slab)
    G.set_stage_variant(variant)
    G.set_state(S)
    assert O.coarse_step() == G.coarse_step()
    np.testing.assert_array_equal(G.state(), O.state())
    G.run(1, use_graph=True)
    O.coarse_step()
    assert (G.dt, G.time) == (O.dt, O.time)
    np.testing.assert_array_equal(G.state(), O.state())
    G.close()
