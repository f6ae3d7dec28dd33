"""The species stage of the fused step (K_species): all thirteen species of a
moving, mixed flow, bit for bit against the oracle, at the sizes where its
tiles of 14 x 14 columns and its chunks of planes begin, end or leave a
remainder, for both boundaries, whole and in z-slabs."""
import numpy as np
import pytest

import minicastro as mc
from minicastro import configs
from helpers import oracle_level, small_cfg, table_bin

pytestmark = pytest.mark.gpu

NVAR, NSPEC = 20, 13
URHO, UMX, UEDEN, UEINT, UTEMP, UFS = 0, 1, 4, 5, 6, 7


@pytest.fixture(scope="module", autouse=True)
def gpu_table():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())


def mixed_flow(n, seed):
    """Random density, velocities of both signs (a third of the cells at rest,
    so that faces with both Riemann weights 1/2 occur), energies and partial
    densities, some species absent."""
    rng = np.random.default_rng(seed)
    S = np.zeros(tuple(n) + (NVAR,), order="F")
    rho = np.exp(rng.uniform(-1.0, 1.0, n))
    e = 3e13 * np.exp(rng.uniform(-1.0, 1.0, n))
    v = rng.standard_normal(tuple(n) + (3,)) * 2e6 * (rng.random(tuple(n) + (1,)) > 0.33)
    X = rng.random(tuple(n) + (NSPEC,)) ** 6 * (rng.random(tuple(n) + (NSPEC,)) > 0.2)
    X[..., 0] += 1e-3
    X /= X.sum(axis=-1, keepdims=True)
    S[..., URHO] = rho
    S[..., UMX:UMX + 3] = rho[..., None] * v
    S[..., UEINT] = rho * e
    S[..., UEDEN] = rho * (e + 0.5 * (v ** 2).sum(axis=-1))
    S[..., UTEMP] = 4e5
    S[..., UFS:] = rho[..., None] * X
    return S


# n_cell around multiples of the tile's 14 interior columns; slab 0: whole
CASES = [((14, 14, 14), 1, 0), ((15, 13, 9), 0, 0), ((29, 15, 6), 1, 0), ((28, 16, 7), 0, 0), ((12, 30, 5), 1, 0),
         ((5, 4, 33), 0, 0), ((4, 5, 4), 1, 0), ((43, 6, 4), 0, 0), ((16, 15, 17), 0, 5), ((15, 16, 17), 1, 4),
         ((9, 8, 7), 0, 1), ((6, 5, 12), 0, 11)]


@pytest.mark.parametrize("n,bc,slab", CASES)
def test_mixed_species_match_oracle(n, bc, slab):
    hi = tuple(v / 16.0 for v in n)
    cfg = small_cfg(n=16, bc=bc)
    cfg.update(n_cell=n, prob_hi=hi, boxes=configs.grid_boxes(n, 64))
    S = mixed_flow(n, seed=sum(n) + bc)
    O = oracle_level(cfg, nthreads=8)
    O.set_state(S)
    G = mc.Level(n, cfg["boxes"], cfg["prob_lo"], hi, bc, mc.MODE_FUSED)
    G.set_fused_slab(slab)
    G.set_state(S)
    for step in range(2):
        dto, dtg = O.coarse_step(), G.coarse_step()
        assert dtg == dto, (step, dtg, dto)
        np.testing.assert_array_equal(G.state(), O.state(), err_msg="step %d" % step)
    G.run(2, use_graph=True)
    O.coarse_step()
    O.coarse_step()
    assert (G.dt, G.time) == (O.dt, O.time)
    np.testing.assert_array_equal(G.state(), O.state())
    G.close()
