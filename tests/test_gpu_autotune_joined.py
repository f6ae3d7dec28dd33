"""The autotuner on a level whose transverse and final fluxes are joined: state,
clock and later steps unchanged, and of the joined kernel the time of a launch."""
import numpy as np
import pytest

import minicastro as mc
from minicastro import configs
from helpers import small_cfg, table_bin
from test_gpu_species import mixed_flow

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bc,slab", [((62, 60, 57), 1, 0), ((61, 59, 64), 0, 58)])
def test_autotune_of_a_joined_level(n, bc, slab):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())
    cfg = small_cfg(n=16, bc=bc)
    hi = tuple(v / 16.0 for v in n)
    S = mixed_flow(n, seed=sum(n))
    A, B = (mc.Level(n, configs.grid_boxes(n, 64), cfg["prob_lo"], hi, bc, mc.MODE_FUSED) for _ in range(2))
    for L in (A, B):
        L.set_fused_slab(slab)
        L.set_state(S)
        L.run(2)
    S1, c1 = A.state(), (A.steps, A.dt, A.time)
    tuned = A.autotune(reps=5)
    assert (A.steps, A.dt, A.time) == c1
    np.testing.assert_array_equal(A.state(), S1)
    if not slab:  # the default variant's joined kernel, timed in a step
        B.run_timed(1)
        ms, nl = B.run_timed(5)["trans1c"]
        assert tuned["trans1c"][1] > 0.6 * ms / nl
        A.run(6)
    else:
        A.run(3)
        B.run(3)
    assert (A.steps, A.dt, A.time) == (B.steps, B.dt, B.time)
    np.testing.assert_array_equal(A.state(), B.state())
    A.close()
    B.close()
