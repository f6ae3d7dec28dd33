"""Calls that read the EOS table report an error, and launch nothing, while no
table is loaded."""
import ctypes as C

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


def test_backward_pass_with_kept_intermediates(no_table):
    import torch
    cfg = small_cfg(n=8, bc=1, r_init=0.3)
    G = mc.Level(cfg["n_cell"], cfg["boxes"], cfg["prob_lo"], cfg["prob_hi"], cfg["bc"], mc.MODE_PLAIN)
    G.init_data(**cfg)
    U0 = torch.from_numpy(np.ascontiguousarray(G.state().transpose(3, 2, 1, 0))).cuda()
    UN, gN, g0 = torch.empty_like(U0), torch.ones_like(U0), torch.zeros_like(U0)
    A = mc.Adjoint(cfg["n_cell"], cfg["prob_lo"], cfg["prob_hi"], cfg["bc"], 2)
    A.keep_intermediates(True)
    A.forward(U0.data_ptr(), UN.data_ptr(), 2)
    rc, err = no_table(mc.lib().mc_adjoint_backward, A.h, C.c_void_p(gN.data_ptr()), C.c_void_p(g0.data_ptr()))
    assert rc != 0 and "EOS table" in err
    assert not g0.any()
    A.backward(gN.data_ptr(), g0.data_ptr())
    assert g0.any() and torch.isfinite(g0).all()
    A.close()
    G.close()
