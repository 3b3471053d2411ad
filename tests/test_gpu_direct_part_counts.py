"""The direct operator where its sources stay whole, go in a few parts or in many
(nbody.hip, count_parts): few targets, one chunk, chunks that fill the chip or not, in both
precisions and both directions, against the oracle; and without allocation, equal bit for bit
to the handle's own buffers."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


# targets x sources: mostly whole (10 x 1000, 130 x 40, 20000 x 300), a few parts (16384 x 300,
# 40000 x 1000), tens of them (1 x 60000, 128 x 2000, 384 x 20000)
@pytest.mark.parametrize("n_obs,n_src", [(10, 1000), (130, 40), (20000, 300), (16384, 300), (40000, 1000), (1, 60000),
                                         (128, 2000), (384, 20000)])
@pytest.mark.parametrize("kid", [1, 3, 6])
def test_part_counts_match_oracle(tbem, orc, kid, n_obs, n_src):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(n_obs + kid)
    nrm = lambda m: (lambda v: v / np.linalg.norm(v, axis=1)[:, None])(rng.standard_normal((m, 3)))
    obs, on, src, sn, w = rng.uniform(0, 1, (n_obs, 3)), nrm(n_obs), rng.uniform(0, 1, (n_src, 3)), nrm(
        n_src), rng.uniform(0.5, 1.5, n_src)
    R = 1 if kid == 1 else 3
    x, g = rng.standard_normal(R * n_src), rng.standard_normal(R * n_obs)
    print(f"CASE part counts kid={kid} {n_obs}x{n_src}", flush=True)
    data, K = tbem.NBodyData(obs, on, src, sn, w), tbem.make_kernel(kid, 1.0, 0.25)
    ref = orc.direct(kid, obs, on, src, sn, w, x, parallel=True)
    adj = orc.direct_adjoint(kid, obs, on, src, sn, w, g)
    # FP64: a few ulp a pair; a lone target's sum of 60,000 signed terms may cancel to a
    # hundredth of its parts. FP32 pairs: 2e-6 likewise
    for precision, tol in (("fp64", 1e-12), ("mixed", 2e-5)):
        op = tbem.make_direct_nbody_operator(data, K, precision=precision)
        assert rel_err(op.apply(x), ref) < tol
        assert rel_err(op.apply_adjoint(g), adj) < tol
        d_x = torch.tensor(x, device="cuda")
        y, z = op.apply(d_x), torch.full((R * n_obs,), np.nan, dtype=torch.float64, device="cuda")
        op.apply_noalloc(d_x, z)
        assert np.array_equal(y.cpu().numpy().view(np.uint64), z.cpu().numpy().view(np.uint64))
