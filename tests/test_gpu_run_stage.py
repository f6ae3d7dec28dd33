"""Single stages after a step that joined its transverse and final fluxes: the
final stage makes the fluxes it reads, and the update that follows equals that of
an engine whose step left them in memory."""
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


@pytest.mark.parametrize("bc,how,final", [(1, "advance", "final"), (0, "graph", "finalc"), (1, "timed", "finalc"),
                                          (0, "eager", "final"), (1, "autotune", "final")])
def test_final_and_update_after_a_joined_step(bc, how, final):
    n = (61, 58, 60)
    cfg = small_cfg(n=16, bc=bc)
    hi = tuple(v / 16.0 for v in n)
    S = mixed_flow(n, seed=11 + bc)
    states = []
    for variant in (0, 2):  # joined; FACE_TRANS1
        L = mc.Level(n, configs.grid_boxes(n, 64), cfg["prob_lo"], hi, bc, mc.MODE_FUSED)
        L.set_stage_variant(variant)
        L.set_state(S)
        L.run(1, use_graph=False)
        if how == "advance":
            L.advance(1e-9)
        elif how == "timed":
            L.run_timed(1)
        else:
            L.run(2, use_graph=how == "graph")
        if how == "autotune":  # leaves the arrays of the step after the state
            L.autotune(reps=1)
            L.set_stage_variant(variant)
        for _ in range(2):
            L.run_stage(L.STAGES.index(final))
        L.run_stage(L.STAGES.index("update"))
        L.run(1)
        states.append(L.state())
        L.close()
    assert np.isfinite(states[1]).all()
    np.testing.assert_array_equal(states[0], states[1])
