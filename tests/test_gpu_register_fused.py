"""Flux registers fed by the fused engine's final fluxes: the same bits as from
the per-box path's, for a mixed flow, unequal refinement ratios and both
boundaries."""
import numpy as np
import pytest

import minicastro as mc
from minicastro import amr, configs
from helpers import table_bin
from test_gpu_species import mixed_flow

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ratio,bc", [((2, 2, 2), 1), ((4, 2, 1), 0), ((1, 3, 2), 1), ((2, 1, 4), 0)])
def test_registers_match_per_box_levels(ratio, bc):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())
    nc = (12, 10, 8)
    nf = tuple(a * b for a, b in zip(nc, ratio))
    box = np.array(nf) // 2  # eight fine boxes, three of them refined
    fine = np.array([[i * box[0], j * box[1], k * box[2], (i + 1) * box[0] - 1, (j + 1) * box[1] - 1,
                      (k + 1) * box[2] - 1] for k in range(2) for j in range(2) for i in range(2)], dtype=np.int32)
    region = [0, 3, 6]
    hi = tuple(v / 16.0 for v in nc)
    Sc, Sf = mixed_flow(nc, seed=sum(ratio)), mixed_flow(nf, seed=40 + bc)
    data = []
    for mode in (mc.MODE_PLAIN, mc.MODE_FUSED):
        Gc = mc.Level(nc, configs.grid_boxes(nc, 64), (0.0, 0.0, 0.0), hi, bc, mode)
        Gf = mc.Level(nf, fine, (0.0, 0.0, 0.0), hi, bc, mode)
        R = amr.FluxRegister(fine[region], ratio, nc, bc)
        amr.set_flux_registers(Gc, crse_side=R)
        amr.set_flux_registers(Gf, fine_side=R)
        Gc.set_state(Sc)
        Gf.set_state(Sf)
        Gc.advance(2e-10)
        data.append([R.data()])
        for _ in range(2):
            Gf.advance(1e-10)
            Gf.post_timestep()
            data[-1].append(R.data())
        data[-1].append(Gf.state())
    for a, b in zip(*data):
        assert np.isfinite(a).all() and (a != 0).any()
        np.testing.assert_array_equal(a, b)
