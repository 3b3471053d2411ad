"""The surface stages above 64 surface points at the edges of their shapes: slices per target
(three up to 84 points, two to 128, one above), parts of 64 targets (three and four, even and
uneven), and the general kernel again past 256 points. Laplace, and the elastic kernels up to
128 points, take one workgroup per item (k_surf_one), the elastic kernels of these small
problems above that several (k_surf_split). Against the
oracle FMM on its own check-to-equivalent matrices, so that neither the method's error nor
another pseudo-inverse enters; the transpose by its identity.

Tolerance: the two sides round a check potential's sum differently, by some 1e-15, and the
check-to-equivalent matrices amplify that, 1e4 times at 75 points; 1e7 is allowed for 258. A
source left out of a sum, or added twice, shows at 1e-4 and more."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def order_of(tbem, n_e):
    for order in range(n_e - 3, n_e + 4):
        if tbem.surface_points(order).shape[0] == n_e:
            return order
    raise AssertionError(f"no order has {n_e} surface points")


@pytest.mark.parametrize("kid,n_e", [(0, 65), (0, 84), (1, 86), (0, 128), (1, 130), (0, 192), (0, 254), (0, 256), (1, 258),
                                     (3, 65), (3, 84), (4, 86), (5, 128), (4, 130), (6, 130), (5, 192), (3, 196),
                                     (4, 198), (3, 256), (4, 258)])
def test_surface_stages_match_oracle(tbem, orc, kid, n_e):
    order = order_of(tbem, n_e)
    rng = np.random.default_rng(order + kid)
    n, m, R = 700, 601, 1 if kid < 2 else 3
    nrm = lambda k: (lambda v: v / np.linalg.norm(v, axis=1)[:, None])(rng.standard_normal((k, 3)))
    src, obs = rng.uniform(0, 1, (n, 3)), rng.uniform(0, 1, (m, 3)) * [1, 1, 0.2]
    sn, on, w = nrm(n), nrm(m), rng.uniform(0.5, 1.5, n)
    x, g = rng.standard_normal(R * n), rng.standard_normal(R * m)
    print(f"CASE surface stages kid={kid} order={order} n_e={n_e}", flush=True)
    of = orc.fmm(kid, obs, on, src, sn, w, 0.3, order, 20, 0.05, False)
    c = of.counts()
    up = np.array([of.c2e(False, L) for L in range(c["n_up_levels"])])
    down = np.array([of.c2e(True, L) for L in range(c["n_down_levels"])])
    op = tbem.FMMOperator(tbem.make_kernel(kid, 1.0, 0.25), tbem.NBodyData(obs, on, src, sn, w),
                          tbem.FMMConfig(0.3, order, 20, 0.05, False), up_c2e=up, down_c2e=down)
    info = op.info()
    assert info["n_e"] == n_e and info["m2l"] == c["m2l"] > 500 and info["m2l_classes"] == 0
    y = op.apply(x)
    assert rel_err(y, of.apply(x)) < 1e-8
    xt = op.apply_adjoint(g)
    scale = np.abs(y).max() * np.abs(g).sum() + np.abs(x).max() * np.abs(xt).sum()
    assert abs(y @ g - x @ xt) < 1e-9 * scale
    assert np.array_equal(op.apply(x), y) and np.array_equal(op.apply_adjoint(g), xt)
