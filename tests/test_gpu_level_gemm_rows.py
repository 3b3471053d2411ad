"""The per-level products (k_level_gemm), which serve operators of 48 rows and more: row counts
below, at and past the edges of their 16- and 64-row tiles, M and its transpose, in the form
for few cells against the oracle FMM on its own check-to-equivalent matrices (tolerances as in
test_gpu_surf_edges), and in the form for many cells, with FP64 and FP32 results, against the
direct sum: there a row or a cell left out shows at 1e-3 and more, the method's error and the
mixed path's rounding are below 1e-4."""
import numpy as np
import pytest

from conftest import rel_err
from test_gpu_surf_edges import order_of

pytestmark = pytest.mark.gpu


def points(n, seed):
    rng = np.random.default_rng(seed)
    nrm = rng.standard_normal((n, 3))
    return rng, rng.uniform(0, 1, (n, 3)), nrm / np.linalg.norm(nrm, axis=1)[:, None], rng.uniform(0.5, 1.5, n)


# (Laplace from 128 rows on: one unit in the last place of the check-to-equivalent matrices moves
# the result by 1.8e-8, more than a test against the oracle can tell from a fault of one cell)
@pytest.mark.parametrize("kid,n_e", [(0, 48), (0, 50), (0, 64), (0, 65), (0, 67), (3, 18), (3, 20), (3, 22), (4, 44)])
def test_few_cells_match_oracle(tbem, orc, kid, n_e):
    order, R, n = order_of(tbem, n_e), 1 if kid < 2 else 3, 2000
    rng, locs, nrm, w = points(n, n_e)
    x, g = rng.standard_normal(R * n), rng.standard_normal(R * n)
    print(f"CASE level products, few cells kid={kid} rows={R * n_e}", flush=True)
    of = orc.fmm(kid, locs, nrm, locs, nrm, w, 0.3, order, 30, 0.05, False)
    c = of.counts()
    up = np.array([of.c2e(False, L) for L in range(c["n_up_levels"])])
    down = np.array([of.c2e(True, L) for L in range(c["n_down_levels"])])
    op = tbem.FMMOperator(tbem.make_kernel(kid, 1.0, 0.25), tbem.NBodyData(locs, nrm, locs, nrm, w),
                          tbem.FMMConfig(0.3, order, 30, 0.05, False), up_c2e=up, down_c2e=down)
    assert op.info()["n_e"] == n_e and R * n_e >= 48 and op.info()["m2l"] > 200
    y = op.apply(x)
    assert rel_err(y, of.apply(x)) < 1e-8
    xt = op.apply_adjoint(g)
    scale = np.abs(y).max() * np.abs(g).sum() + np.abs(x).max() * np.abs(xt).sum()
    assert abs(y @ g - x @ xt) < 1e-9 * scale


# at least 512 workgroups: 64-row tiles times 64-cell tiles of the leaves
@pytest.mark.parametrize("kid,n_e,n", [(0, 64, 120000), (0, 65, 100000), (0, 130, 60000), (3, 44, 50000)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_many_cells_match_direct_sum(tbem, kid, n_e, n, precision):
    order, R = order_of(tbem, n_e), 1 if kid < 2 else 3
    rng, locs, nrm, w = points(n, n_e)
    x, g = rng.uniform(0.5, 1.5, R * n), rng.uniform(0.5, 1.5, R * n)
    print(f"CASE level products, many cells kid={kid} rows={R * n_e} n={n} {precision}", flush=True)
    K, data = tbem.make_kernel(kid, 1.0, 0.25), tbem.NBodyData(locs, nrm, locs, nrm, w)
    op = tbem.FMMOperator(K, data, tbem.FMMConfig(0.3, order, 4, 0.05, False), precision)
    info = op.info()
    tiles = -(-(R * n_e) // 64) * (info["p2m"] // 64)
    assert info["n_e"] == n_e and tiles >= 512
    direct = tbem.make_direct_nbody_operator(data, K)
    assert rel_err(op.apply(x), direct.apply(x)) < 1e-4
    assert rel_err(op.apply_adjoint(g), direct.apply_adjoint(g)) < 1e-4
