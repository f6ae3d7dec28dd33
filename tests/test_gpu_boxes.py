"""The per-box path's kernels over several boxes at once (clean_state,
FillPatch) and the finish of its fluxes: bit for bit against the oracle, for
uneven boxes down to one cell thick, with densities under the floor, negative
energies and cells at rest, for both boundaries."""
import numpy as np
import pytest

import minicastro as mc
from helpers import oracle_level, small_cfg, table_bin
from test_gpu_species import UEDEN, UEINT, UFS, UMX, URHO, mixed_flow

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu_table():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())


def split(n, cuts):
    """Boxes (lo, hi) of the tensor product of the cuts of each direction."""
    e = [[0] + list(c) + [m] for c, m in zip(cuts, n)]
    return np.array([[e[0][i], e[1][j], e[2][k], e[0][i + 1] - 1, e[1][j + 1] - 1, e[2][k + 1] - 1]
                     for k in range(len(e[2]) - 1) for j in range(len(e[1]) - 1) for i in range(len(e[0]) - 1)],
                    dtype=np.int32)


@pytest.mark.parametrize("n,cuts,bc,floors", [((17, 9, 6), ((1, 10), (4,), ()), 1, False),
                                              ((8, 21, 7), ((), (16,), (1, 2)), 0, False),
                                              ((17, 9, 6), ((1, 10), (4,), ()), 0, True),
                                              ((6, 5, 4), ((), (), ()), 1, True)])
def test_uneven_boxes_match_oracle(n, cuts, bc, floors):
    hi = tuple(v / 16.0 for v in n)
    boxes = split(n, cuts)
    cfg = small_cfg(n=16, bc=bc)
    cfg.update(n_cell=n, prob_hi=hi, boxes=boxes)
    S = mixed_flow(n, seed=sum(n) + bc)
    if floors:
        for c in ((0, 0, 0), (n[0] - 1, 2, 1)):  # under the density floor
            S[c] *= 1e-40 / S[c][URHO]
        S[3, 1, 2, UEINT] = -S[3, 1, 2, UEINT]
        S[4, 2, 1, UEDEN] = -S[4, 2, 1, UEDEN]
    S[2, 3, 3, UMX:UMX + 3] = 0.0
    S[1, 1, 1, UFS:] *= 0.5  # species that do not sum to the density
    O = oracle_level(cfg, nthreads=8)
    O.set_state(S)
    G = mc.Level(n, boxes, cfg["prob_lo"], hi, bc, mc.MODE_PLAIN)
    G.set_state(S)
    for step in range(2):
        dto, dtg = O.coarse_step(), G.coarse_step()
        assert dtg == dto, (step, dtg, dto)
        np.testing.assert_array_equal(G.state(), O.state(), err_msg="step %d" % step)
    G.close()
