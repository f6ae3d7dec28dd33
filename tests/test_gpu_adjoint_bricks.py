"""The bricks of the adjoint's reverse kernels: the gradient against the CPU
tangent-linear (test_gpu_adjoint, same bound) on cubes whose sides are shorter
than a brick, fill it exactly or leave a remainder, for both boundaries."""
import pytest

from test_gpu_adjoint import gpu_table, tangent_check  # noqa: F401 (gpu_table: fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bc", [(5, 1), (6, 0), (14, 0), (17, 1), (30, 1), (31, 0)])
def test_brick_edges_match_cpu_tangent_linear(n, bc):
    assert max(tangent_check(n, 2, 2, seed=n, bc=bc, r_init=0.3, shell=(0.1, 0.6))) < 1e-10
