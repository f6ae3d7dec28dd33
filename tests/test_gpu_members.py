"""Ensembles of more members than a workgroup has threads: the last ones step
as the first do."""
import numpy as np
import pytest

import minicastro as mc
from minicastro import configs
from helpers import table_bin

pytestmark = pytest.mark.gpu


def test_members_past_the_first_workgroup_step():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mc.load_table(table_bin())
    one = dict(configs.UNIT_SEDOV, n_cell=(4, 4, 4), boxes=configs.grid_boxes(4, 4), r_init=0.3)
    E = mc.Ensemble([dict(one) for _ in range(300)])
    E.init_data()
    E.run(2)
    first = E.clock(0)
    assert first[2] == 2 and first[0] > 0.0
    for m in (255, 256, 299):
        assert E.clock(m) == first
        np.testing.assert_array_equal(E.state(m), E.state(0))
    E.close()
