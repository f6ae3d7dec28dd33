"""Limits of the fused engine's 32-bit offsets that need no device memory to
meet: refusals come before any of it is taken."""
import ctypes as C

import pytest

import minicastro as mc
from helpers import table_bin

pytestmark = pytest.mark.gpu


# wide, shallow instances whose face arrays fit but whose primitives' planes
# do not: a ring of 9 planes, of 11, and whole (no deeper than the ring)
@pytest.mark.parametrize("n,slab", [((5500, 5500, 14), 1), ((4950, 4950, 20), 3), ((5200, 5200, 10), 6)])
def test_primitives_beyond_their_offsets_are_refused(n, slab):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())
    assert (n[0] + 2) * (n[1] + 2) * (slab + 2) < 2 ** 28 and n[0] * n[1] * n[2] < 2 ** 29
    assert n[0] * n[1] * min(n[2], slab + 8) >= 2 ** 28
    free = torch.cuda.mem_get_info()[0]
    with pytest.raises(RuntimeError, match="primitives.*2\\^28"):
        mc.Ensemble([dict(n_cell=n, prob_lo=(0, 0, 0), prob_hi=(1, 1, 1), bc=1, p_ambient=1e13, dens_ambient=1.0,
                          exp_energy=1e12, r_init=0.1)], slab=slab)
    assert torch.cuda.mem_get_info()[0] > free - 2 ** 28


def test_shallow_instance_below_the_limit_keeps_whole_primitives():
    """5500 x 5500 x 4 in slabs of one plane: a ring of nine planes would pass
    2^28 cells, the four there are do not."""
    n = (C.c_int * 3)(5500, 5500, 4)
    cells = 5500 * 5500 * 4
    assert 8 * 50 * cells <= mc.lib().mc_fused_bytes(1, n, 1) < 8 * (50 * cells + 200 * 5502 * 5502 * 3)
