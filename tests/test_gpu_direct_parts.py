"""The direct operator's source parts (nbody.hip, split_sources): one part and many, the
last one short or of a single source, one target, whole and ragged target chunks."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def point_set(n_obs, n_src, seed):
    rng = np.random.default_rng(seed)
    nrm = lambda m: (lambda v: v / np.linalg.norm(v, axis=1)[:, None])(rng.standard_normal((m, 3)))
    return rng, rng.uniform(0, 1, (n_obs, 3)), nrm(n_obs), rng.uniform(0, 1, (n_src, 3)), nrm(n_src), rng.uniform(
        0.5, 1.5, n_src)


@pytest.mark.parametrize("n_obs,n_src", [(1, 1), (1, 65), (127, 64), (128, 4097), (129, 513), (300, 5000), (2003, 3000)])
@pytest.mark.parametrize("kid", [0, 1, 4, 6])
def test_direct_parts_match_oracle(tbem, orc, kid, n_obs, n_src):
    rng, obs, on, src, sn, w = point_set(n_obs, n_src, 5 + kid)
    R = 1 if kid < 2 else 3
    x, g = rng.standard_normal(R * n_src), rng.standard_normal(R * n_obs)
    print(f"CASE direct parts kid={kid} {n_obs}x{n_src}", flush=True)
    data, K = tbem.NBodyData(obs, on, src, sn, w), tbem.make_kernel(kid, 1.0, 0.25)
    op = tbem.make_direct_nbody_operator(data, K)
    ref = orc.direct(kid, obs, on, src, sn, w, x, parallel=True)
    adj = orc.direct_adjoint(kid, obs, on, src, sn, w, g)
    assert rel_err(op.apply(x), ref) < 1e-13
    assert rel_err(op.apply_adjoint(g), adj) < 1e-13
    mixed = tbem.make_direct_nbody_operator(data, K, precision="mixed")
    assert rel_err(mixed.apply(x), ref) < 2e-6  # FP32 pairs: a few ulp each, summed without cancellation control
    assert rel_err(mixed.apply_adjoint(g), adj) < 2e-6
