"""The one-target-per-lane surface stage (k_surf_one) at the edges of its range of surface
points and slices (65, 84 | 85, 128 | 129, 256 | 257), forward and transpose, on distinct
point sets, whose M2L runs on surfaces. Against the direct sum: at these orders the method's
error is below 1e-5, a wrong target or source shows at its full size."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kid,order", [(0, 65), (0, 84), (1, 85), (0, 128), (1, 129), (0, 256), (0, 257), (3, 66),
                                       (4, 100), (5, 85), (3, 150)])
def test_surface_stage_matches_direct_sum(tbem, kid, order):
    rng = np.random.default_rng(order)
    n, m, R = 5000, 4001, 1 if kid < 2 else 3
    nrm = lambda k: (lambda v: v / np.linalg.norm(v, axis=1)[:, None])(rng.standard_normal((k, 3)))
    src, obs = rng.uniform(0, 1, (n, 3)), rng.uniform(0, 1, (m, 3)) * [1, 1, 0.2]
    data, K = tbem.NBodyData(obs, nrm(m), src, nrm(n), rng.uniform(0.5, 1.5, n)), tbem.make_kernel(kid, 1.0, 0.25)
    x, g = rng.standard_normal(R * n), rng.standard_normal(R * m)
    n_e = tbem.surface_points(order).shape[0]
    print(f"CASE surface stage kid={kid} order={order} n_e={n_e}", flush=True)
    op, direct = tbem.FMMOperator(K, data, tbem.FMMConfig(0.3, order, 40, 0.05, False)), tbem.make_direct_nbody_operator(
        data, K)
    assert op.info()["m2l"] > 1000 and op.info()["m2l_classes"] == 0
    assert rel_err(op.apply(x), direct.apply(x)) < 1e-4
    assert rel_err(op.apply_adjoint(g), direct.apply_adjoint(g)) < 1e-4
