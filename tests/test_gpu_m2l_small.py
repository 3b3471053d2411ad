"""The FP64 class M2L at operator sizes below 48 rows (one to three row tiles), against the
surfaces' evaluation of the same pairs: both directions, the gradient, FP64 and mixed
precision; and the sizes that stay on the surfaces."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def pair_of_ops(tbem, kid, n, order, precision):
    rng = np.random.default_rng(order)
    locs, nrm = rng.uniform(0, 1, (n, 3)), rng.standard_normal((n, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    K, data = tbem.make_kernel(kid, 1.0, 0.25), tbem.NBodyData(locs, nrm, locs, nrm, rng.uniform(0.5, 1.5, n))
    cfg = tbem.FMMConfig(0.3, order, 60, 0.05, False)
    return K, [tbem.FMMOperator(K, data, cfg, precision, translations=t) for t in ("auto", "surfaces")]


# agreement: 1e-12 up to order 20, and the C2E's amplification of last-bit differences above
# (4e-11 at order 50 with Laplace), as between the two forms at larger sizes
@pytest.mark.parametrize("kid,order,tol", [(0, 16, 1e-11), (0, 17, 1e-11), (0, 32, 1e-9), (0, 35, 1e-9), (0, 44, 1e-9),
                                           (1, 20, 1e-11), (1, 33, 1e-9), (6, 10, 1e-11)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_small_class_operators_match_surfaces(tbem, kid, order, tol, precision):
    print(f"CASE small classes kid={kid} order={order} {precision}", flush=True)
    K, (a, b) = pair_of_ops(tbem, kid, 12000, order, precision)
    assert K.dim * a.info()["n_e"] < 48 and a.info()["m2l_classes"] > 0 and b.info()["m2l_classes"] == 0
    rng = np.random.default_rng(2)
    x, g = rng.standard_normal(12000 * K.dim), rng.standard_normal(12000 * K.dim)
    ya, yb = a.apply(x), b.apply(x)
    assert rel_err(ya, yb) < tol
    assert rel_err(a.apply_adjoint(g), b.apply_adjoint(g)) < tol
    assert rel_err(a.obs_grad(x, g), b.obs_grad(x, g)) < 10 * tol
    assert np.array_equal(a.apply(x), ya)


@pytest.mark.parametrize("kid,n,order", [(0, 12000, 5), (3, 12000, 6), (0, 500, 35)])
def test_sizes_that_stay_on_the_surfaces(tbem, kid, n, order):
    K, (a, _) = pair_of_ops(tbem, kid, n, order, "fp64")
    assert a.info()["m2l_classes"] == 0
