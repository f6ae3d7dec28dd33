"""Calls that read the EOS table report an error, and launch nothing, while no
table is loaded."""
import numpy as np
import pytest

import minicastro as mc
from helpers import small_cfg, table_bin

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu_table():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())


@pytest.fixture
def no_table():
    """Calls made through it run without a table."""
    def call(f, *args):
        mc.lib().eos_finalize()
        try:
            return f(*args), mc.lib().mc_last_error().decode()
        finally:
            mc.load_table(table_bin())
    return call


def test_post_timestep_of_a_per_box_level(no_table):
    cfg = small_cfg(n=16, bc=1)
    L = mc.Level(cfg["n_cell"], cfg["boxes"], cfg["prob_lo"], cfg["prob_hi"], cfg["bc"], mc.MODE_PLAIN)
    L.init_data(**cfg)
    L.advance(0.5 * L.est_time_step())
    S = L.state()
    rc, err = no_table(mc.lib().mc_level_post_timestep, L.h)
    assert rc != 0 and "EOS table" in err
    np.testing.assert_array_equal(L.state(), S)
    L.post_timestep()
    L.close()
