"""A coarse step made of the drop-in entry points alone, called box by box in the
order of Castro::advance and construct_hydro_source (Source/Castro_advance.cpp:
11-100, Source/Castro_hydro.cpp:31-397), as a reference host calls them: bit for
bit the oracle's step."""
import numpy as np
import pytest

import orc
import minicastro as mc
from helpers import Dev, NGDNV, NQAUX, NVAR, QVAR, gpu_call, oracle_level, small_cfg, table_bin
from test_gpu_kernels import grow, grow3, nodes, sub
from test_gpu_species import UEDEN, UEINT, URHO, mixed_flow

pytestmark = pytest.mark.gpu

# how far a direction's states reach beyond its faces: traced, and corrected by
# the transverse fluxes of direction e
REACH = {(0, 0): (0, 1, 1), (0, 1): (0, 0, 1), (0, 2): (0, 1, 0), (1, 0): (0, 0, 1), (1, 1): (1, 0, 1),
         (1, 2): (1, 0, 0), (2, 0): (0, 1, 0), (2, 1): (1, 0, 0), (2, 2): (1, 1, 0)}


def clean_state(s):
    for name in ("enforce_minimum_density", "normalize_species", "reset_internal_e", "compute_temp"):
        gpu_call(name, orc.iv(*s.lo), orc.iv(*s.hi), s)


def hydro_source(state, bx, n, dx, dt):
    """The hydro source of a box from its S_border FAB, and the fluxes store_flux
    writes."""
    lo, hi = bx
    dxv, iv = orc.dv(*dx), lambda b: (orc.iv(*b[0]), orc.iv(*b[1]))
    qbx, obx = grow(lo, hi, 4), grow(lo, hi, 1)
    ebx = [nodes(lo, hi, d) for d in range(3)]
    gebx = [grow(*e, 1) for e in ebx]
    tbx = {k: grow3(*ebx[k[0]], r) for k, r in REACH.items()}
    area = [Dev(*b, 1, np.full(tuple(h - l + 1 for l, h in zip(*b)), np.prod(dx) / dx[d]))
            for d, b in enumerate(grow(*e, 4) for e in ebx)]
    vol = Dev(*qbx, 1, np.full(tuple(h - l + 1 for l, h in zip(*qbx)), dx[0] * dx[1] * dx[2]))
    q, qaux, div = Dev(*qbx, QVAR), Dev(*qbx, NQAUX), Dev(*obx, 1)
    gpu_call("ctoprim", *iv(qbx), state, q, qaux)
    gpu_call("divu", *iv(obx), q, dxv, div)
    hdt, cdt = [0.5 * dt / v for v in dx], [dt / v / 3.0 for v in dx]
    qm, qp = {k: Dev(*b, QVAR) for k, b in tbx.items()}, {k: Dev(*b, QVAR) for k, b in tbx.items()}
    q_int, f1, f2, g1, g2 = Dev(*obx, QVAR), Dev(*obx, NVAR), Dev(*obx, NVAR), Dev(*obx, NGDNV), Dev(*obx, NGDNV)
    for d in range(3):
        gpu_call("trace_ppm", *iv(obx), *iv(bx), d + 1, q, qaux, qm[d, d], qp[d, d], orc.iv(0, 0, 0),
                 orc.iv(*[v - 1 for v in n]), dxv, dt)
    across = [(1, 2), (0, 2), (0, 1)]
    for d in range(3):
        gpu_call("compute_flux", *iv(tbx[d, d]), qm[d, d], qp[d, d], f1, q_int, g1, qaux, d + 1)
        for t in across[d]:
            gpu_call("trans1", *iv(tbx[t, d]), d + 1, t + 1, qm[t, t], qm[t, d], qp[t, t], qp[t, d], qaux, f1, g1,
                     cdt[d])
    flux, qe = [Dev(*b, NVAR) for b in gebx], [Dev(*b, NGDNV) for b in gebx]
    ql, qr = Dev(*obx, QVAR), Dev(*obx, QVAR)
    for d in range(3):
        a, b = across[d]
        gpu_call("compute_flux", *iv(tbx[a, b]), qm[a, b], qp[a, b], f1, q_int, g1, qaux, a + 1)
        gpu_call("compute_flux", *iv(tbx[b, a]), qm[b, a], qp[b, a], f2, q_int, g2, qaux, b + 1)
        gpu_call("trans2", *iv(ebx[d]), d + 1, a + 1, b + 1, qm[d, d], ql, qp[d, d], qr, qaux, f1, f2, g1, g2, hdt[d],
                 hdt[a], hdt[b])
        gpu_call("compute_flux", *iv(ebx[d]), ql, qr, flux[d], q_int, qe[d], qaux, d + 1)
    out = [Dev(*e, NVAR) for e in ebx]
    for d in range(3):
        gpu_call("apply_av", *iv(ebx[d]), d + 1, dxv, div, state, flux[d])
        gpu_call("normalize_species_fluxes", *iv(ebx[d]), flux[d])
        gpu_call("store_flux", *iv(ebx[d]), out[d], flux[d], area[d], dt)
    src = Dev(lo, hi, NVAR, np.zeros(tuple(h - l + 1 for l, h in zip(lo, hi)) + (NVAR,)))
    gpu_call("fill_hydro_source", *iv(bx), state, q, src, *flux, *qe, *area, vol, dxv, dt)
    return src, out


@pytest.mark.parametrize("floors", [False, True])
def test_step_of_entry_points_matches_oracle(floors):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())
    n = (13, 9, 8)
    hi = tuple(v / 16.0 for v in n)
    boxes = [((0, 0, 0), (4, 8, 7)), ((5, 0, 0), (12, 3, 7)), ((5, 4, 0), (12, 8, 7))]
    cfg = small_cfg(n=16, bc=1)
    cfg.update(n_cell=n, prob_hi=hi, boxes=np.array([b[0] + b[1] for b in boxes], dtype=np.int32))
    S = mixed_flow(n, seed=31)
    if floors:
        S[0, 0, 0] *= 1e-40 / S[0, 0, 0, URHO]
        S[6, 5, 2, UEINT] = -S[6, 5, 2, UEINT]
        S[7, 1, 3, UEDEN] = -S[7, 1, 3, UEDEN]
    O = oracle_level(cfg, nthreads=8)
    O.set_state(S)
    dt = O.coarse_step()
    at = lambda b: tuple(slice(l, h + 1) for l, h in zip(*b))
    old = [Dev(*b, NVAR, S[at(b)]) for b in boxes]
    for s in old:
        clean_state(s)
    whole = np.empty(n + (NVAR,), order="F")
    for b, s in zip(boxes, old):
        whole[at(b)] = s.host()
    got, faces = np.empty_like(whole), {}
    for b in boxes:
        border = Dev(*grow(*b, 4), NVAR, sub(whole, *grow(*b, 4)))  # FillPatch
        clean_state(border)
        src, out = hydro_source(border, b, n, (1.0 / 16,) * 3, dt)
        new = Dev(*b, NVAR, whole[at(b)] + dt * src.host())
        clean_state(new)
        clean_state(new)  # post_timestep
        got[at(b)] = new.host()
        for d in range(3):
            faces[b, d] = out[d].host()
    np.testing.assert_array_equal(got, O.state())
    # the boxes that share faces in y store the same fluxes on them
    a, c = faces[boxes[1], 1], faces[boxes[2], 1]
    np.testing.assert_array_equal(a[:, -1], c[:, 0])


def test_ctoprim_of_a_large_box_equals_small_ones():
    """A box of more cells than the kernel for one wavefront per SIMD takes, and
    the same cells in smaller boxes of the same FABs."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())
    n = (47, 40, 36)
    assert 65536 < np.prod(n) < 2 * 65536
    b = ((0, 0, 0), tuple(v - 1 for v in n))
    u = Dev(*b, NVAR, mixed_flow(n, seed=5))
    clean_state(u)
    got = []
    for cuts in ((0, 47), (0, 20, 47), (0, 1, 30, 47)):
        q, qaux = Dev(*b, QVAR), Dev(*b, NQAUX)
        for lo, hi in zip(cuts, cuts[1:]):
            gpu_call("ctoprim", orc.iv(lo, 0, 0), orc.iv(hi - 1, 39, 35), u, q, qaux)
        got.append((q.host(), qaux.host()))
    for q, qaux in got[1:]:
        np.testing.assert_array_equal(q, got[0][0])
        np.testing.assert_array_equal(qaux, got[0][1])
