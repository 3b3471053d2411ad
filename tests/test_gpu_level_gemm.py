"""The per-level products (k_level_gemm) at the edges of their tiles: operator sizes below,
at and just past 16, 32 and 64 rows, chunks of k that end ragged, and few or many cells per
level, forward and transpose (op(M) = M and M^T), against the oracle FMM."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kid,order,n,leaf", [(0, 5, 40, 4), (0, 16, 3000, 20), (0, 17, 3000, 20), (0, 35, 20000, 4),
                                              (0, 63, 2000, 30), (0, 64, 2000, 30), (3, 21, 2000, 30),
                                              (3, 22, 6000, 12), (4, 6, 30000, 5)])
def test_level_products_match_oracle(tbem, orc, kid, order, n, leaf):
    rng = np.random.default_rng(order + n)
    R = 1 if kid == 0 else 3
    locs, nrm = rng.uniform(0, 1, (n, 3)), rng.standard_normal((n, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    w, x, g = rng.uniform(0.5, 1.5, n), rng.standard_normal(R * n), rng.standard_normal(R * n)
    print(f"CASE level products kid={kid} order={order} n={n} leaf={leaf}", flush=True)
    of = orc.fmm(kid, locs, nrm, locs, nrm, w, 0.3, order, leaf, 0.05, False)
    op = tbem.FMMOperator(tbem.make_kernel(kid, 1.0, 0.25), tbem.NBodyData(locs, nrm, locs, nrm, w),
                          tbem.FMMConfig(0.3, order, leaf, 0.05, False))
    y, ref = op.apply(x), of.apply(x)
    # the C2E amplifies the last bits of the two sides' pseudo-inverses: 1e-12 at low order,
    # 1e4 times a rounding at order 75
    assert rel_err(y, ref) < (1e-12 if order < 16 else 1e-8)
    if order < 16:  # above, the C2E's amplification of a rounding hides in the identity too
        xt = op.apply_adjoint(g)
        scale = np.abs(y).max() * np.abs(g).sum() + np.abs(x).max() * np.abs(xt).sum()
        assert abs(y @ g - x @ xt) < 1e-13 * scale
