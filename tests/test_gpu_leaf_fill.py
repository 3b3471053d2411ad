"""Leaves cut by the problem's size (fmm.hip, split_leaves and build_sym): the small
problems whose items are cut most, with leaves on the one-wave, the one-workgroup and the
symmetric kernels, against the oracle; and mixed precision, whose cuts fall on whole FP32
tiles, against FP64 at its usual distance."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kid,n,leaf", [(0, 300, 100), (0, 3000, 60), (0, 9000, 260), (1, 5000, 130), (3, 700, 64),
                                        (3, 6000, 64), (3, 6000, 250), (3, 4000, 400), (4, 5000, 100), (6, 5000, 65),
                                        (6, 3000, 129)])
def test_cut_leaves_match_oracle(tbem, orc, kid, n, leaf):
    rng = np.random.default_rng(n + kid)
    R = 1 if kid < 2 else 3
    locs = np.vstack([rng.uniform(0, 1, (n - n // 4, 3)), 0.4 + 0.01 * rng.standard_normal((n // 4, 3))])
    nrm = rng.standard_normal((n, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    w, x, g = rng.uniform(0.5, 1.5, n), rng.standard_normal(R * n), rng.standard_normal(R * n)
    print(f"CASE cut leaves kid={kid} n={n} leaf={leaf}", flush=True)
    K, data, cfg = tbem.make_kernel(kid, 1.0, 0.25), tbem.NBodyData(locs, nrm, locs, nrm, w), tbem.FMMConfig(
        0.3, 5, leaf, 0.05, False)
    ref = orc.fmm(kid, locs, nrm, locs, nrm, w, 0.3, 5, leaf, 0.05, False).apply(x)
    op = tbem.FMMOperator(K, data, cfg)
    for overlap in (False, True):
        op.set_overlap(overlap)
        y = op.apply(x)
        assert rel_err(y, ref) < 1e-12
        xt = op.apply_adjoint(g)
        scale = np.abs(y).max() * np.abs(g).sum() + np.abs(x).max() * np.abs(xt).sum()
        assert abs(y @ g - x @ xt) < 1e-13 * scale
    m = tbem.FMMOperator(K, data, cfg, precision="mixed")
    assert rel_err(m.apply(x), ref) < 2e-5 and rel_err(m.apply_adjoint(g), xt) < 2e-5
