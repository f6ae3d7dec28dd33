"""The ring of planes that holds an engine's primitives in slabs: large levels
in slabs, shallow and deep, with a last slab of fewer planes, equal the
whole-level engine bit for bit; which levels keep one."""
import ctypes as C

import numpy as np
import pytest

import minicastro as mc
from minicastro import configs
from helpers import small_cfg, table_bin
from test_gpu_species import UEDEN, UEINT, mixed_flow

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


def nbytes(n, slab):
    return mc.lib().mc_fused_bytes(1, (C.c_int * 3)(*n), slab)


def test_small_levels_keep_whole_primitives():
    """A level of up to 2,000,000 cells holds the state and the primitives whole
    (50 doubles a cell), so that one launch makes them; a larger one holds the
    primitives of the slab's neighbourhood, unless the level is no deeper.  The
    face arrays take less than 200 doubles a cell of the slab and its ring."""
    def face(n, slab):
        return 8 * 200 * (n[0] + 2) * (n[1] + 2) * (slab + 2)
    for n, slab in (((100, 100, 100), 4), ((2000, 1000, 1), 0), ((1000, 1000, 9), 1), ((1000, 1000, 9), 8)):
        whole = 8 * 50 * n[0] * n[1] * n[2]
        assert whole <= nbytes(n, slab) < whole + face(n, slab or n[2])
    for n, slab in (((150, 150, 150), 4), ((420, 360, 14), 1), ((127, 126, 126), 31)):
        planes = 20 * n[2] + 30 * (slab + 8) + 20 * 8
        assert nbytes(n, slab) < 8 * n[0] * n[1] * planes + face(n, slab)


def test_members_with_and_without_rings():
    """Large members before, between and after small ones, periodic and not."""
    members = [((8, 9, 30), 0), ((127, 126, 126), 0), ((30, 20, 40), 1), ((130, 128, 121), 1), ((12, 10, 5), 0)]
    insts = []
    for (n, bc), r in zip(members, (0.2, 0.8, 0.5, 0.7, 0.2)):
        insts.append(small_cfg(n=16, bc=bc, n_cell=n, prob_hi=tuple(v / 32.0 for v in n), r_init=r))
    out = []
    for slab in (0, 20):
        E = mc.Ensemble(insts, slab=slab)
        E.init_data()
        E.run(3)
        out.append([(E.state(m), E.clock(m)) for m in range(len(insts))])
        E.close()
    for m, ((a, ca), (b, cb)) in enumerate(zip(*out)):
        np.testing.assert_array_equal(a, b, err_msg="member %d" % m)
        assert ca == cb and ca[2] == 3


def test_saved_planes_of_periodic_members_only():
    """Outflow and small members, which save no boundary planes, before and
    between periodic ones that do."""
    members = [((130, 128, 121), 1), ((9, 12, 40), 0), ((127, 126, 126), 0), ((131, 126, 122), 1), ((300, 210, 32), 0)]
    insts = [small_cfg(n=16, bc=bc, n_cell=n, prob_hi=tuple(v / 32.0 for v in n), r_init=0.1 + 0.1 * m)
             for m, (n, bc) in enumerate(members)]
    out = []
    for slab in (0, 9):
        E = mc.Ensemble(insts, slab=slab)
        E.init_data()
        E.run(2)
        out.append([(E.state(m), E.clock(m)) for m in range(len(insts))])
        E.close()
    for m, ((a, ca), (b, cb)) in enumerate(zip(*out)):
        np.testing.assert_array_equal(a, b, err_msg="member %d" % m)
        assert ca == cb


def test_unconverged_solves_counted_once():
    """Cells whose solves do not converge, at the periodic boundary in z: their
    images in the ring are not counted again."""
    n = (127, 126, 126)
    hi = tuple(v / 16.0 for v in n)
    cfg = small_cfg(n=16, bc=0)
    S = mixed_flow(n, seed=3)
    for c in ((5, 7, 0), (60, 1, 3), (100, 125, 124), (0, 64, 125), (30, 30, 60)):
        S[c][[UEDEN, UEINT]] = np.inf
    counts, states = [], []
    for slab in (0, 40, 5):
        L = mc.Level(n, configs.grid_boxes(n, 512), cfg["prob_lo"], hi, 0, mc.MODE_FUSED)
        L.set_fused_slab(slab)
        L.set_state(S)
        mc.newton_failures(reset=True)
        L.advance(1e-9)
        L.sync()
        counts.append(mc.newton_failures(reset=True))
        states.append(L.state())
        L.close()
    assert counts[0] > 0 and counts == counts[:1] * 3
    for s in states[1:]:
        np.testing.assert_array_equal(s, states[0])
