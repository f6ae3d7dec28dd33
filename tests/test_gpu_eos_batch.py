"""Batches of EOS evaluations: (rho, p) solves against the oracle, the same bits
from small and large batches, and the table cell of points about the width of
the single-precision logarithm's guard from a grid line."""
import ctypes as C

import numpy as np
import pytest

import orc
import minicastro as mc
from helpers import oracle_table, table_bin

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu_table():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())
    oracle_table()


def batch(mode, rho, T, ev, abar, zbar):
    import torch
    dev = [torch.from_numpy(np.ascontiguousarray(x, dtype=np.float64)).cuda() for x in (rho, T, ev, abar, zbar)]
    n = len(rho)
    out = torch.zeros(10 * n, dtype=torch.float64, device="cuda")
    P = lambda t: C.cast(t.data_ptr(), C.POINTER(C.c_double))
    assert mc.lib().mc_eos_eval_batch(n, mode, *[P(t) for t in dev], P(out)) == 0
    torch.cuda.synchronize()
    return out.cpu().numpy().reshape(n, 10)


def points(n, seed):
    rng = np.random.default_rng(seed)
    rho, T = 10.0 ** rng.uniform(-6, 6, n), 10.0 ** rng.uniform(3.2, 12.5, n)
    abar = rng.choice([4.0, 12.0, 40.0], n)
    return rho, T, T * 10.0 ** rng.uniform(-1.5, 1.5, n), abar, abar * rng.uniform(0.3, 0.5, n)


def test_pressure_solves_match_oracle():
    rho, T, Tg, abar, zbar = points(3000, 8)
    p = batch(1, rho, T, T, abar, zbar)[:, 1]
    p[[5, 700]] = np.nan  # solves that do not converge end where the oracle's do
    p[[6, 2999]] = np.inf
    mc.newton_failures(reset=True)
    o = batch(3, rho, Tg, p, abar, zbar)
    ref = [orc.eos(orc.EOS_RP, r, t, a, z, p=q) for r, t, a, z, q in zip(rho, Tg, abar, zbar, p)]
    np.testing.assert_array_equal(o[:, 0], [r.T for r in ref])
    np.testing.assert_array_equal(o[:, 2], [r.e for r in ref])
    assert mc.newton_failures(reset=True) >= 4


@pytest.mark.parametrize("n", [65537, 131072])
def test_large_batches_equal_small_ones(n):
    rho, T, Tg, abar, zbar = points(n, n)
    rt = batch(1, rho, T, T, abar, zbar)
    for mode, guess, ev in ((1, T, T), (2, Tg, rt[:, 2]), (3, Tg, rt[:, 1])):
        whole = batch(mode, rho, guess, ev, abar, zbar)
        parts = [batch(mode, *(np.array_split(x, 3)[k] for x in (rho, guess, ev, abar, zbar))) for k in range(3)]
        np.testing.assert_array_equal(whole, np.concatenate(parts))


def test_table_cells_near_the_guard():
    """2^-11 of a cell from every grid line of T and of ye * rho, where the
    single-precision logarithm and log10 take turns, and closer."""
    t, d = orc.eos_grid()
    steps = [s * f for f in (2.0 ** -11 * (1 - 1e-2), 2.0 ** -11 * (1 + 1e-2), 1e-4, 1e-3) for s in (-1, 1)]
    around = lambda g: np.concatenate([10.0 ** (np.log10(g[1:-1]) + s / 20.0) for s in steps])
    Tp, dp = around(t), around(d)  # both axes have 20 cells a decade
    rho = np.concatenate([np.full(Tp.size, 2.0), 2.0 * dp])  # ye = 1/2
    T = np.concatenate([Tp, np.full(dp.size, 1.0e7)])
    abar, zbar = np.full(T.size, 4.0), np.full(T.size, 2.0)
    o = batch(1, rho, T, T, abar, zbar)
    ref = [orc.eos(orc.EOS_RT, r, v, 4.0, 2.0) for r, v in zip(rho, T)]
    for col, name in ((8, "iat"), (9, "jat"), (1, "p"), (2, "e")):
        np.testing.assert_array_equal(o[:, col], [getattr(r, name) for r in ref])
