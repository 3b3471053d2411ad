"""Leaves of very many points: the chunk sums that their cutting leaves between the kernels
(fmm.hip, split_leaves) stay within 2 GiB, and the longer chunks give the same sums."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def one_leaf(tbem, K, n):
    rng = np.random.default_rng(n)
    locs, nrm = rng.uniform(0, 1, (n, 3)), rng.standard_normal((n, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    data = tbem.NBodyData(locs, nrm, locs, nrm, rng.uniform(0.5, 1.5, n))
    return data, tbem.FMMOperator(K, data, tbem.FMMConfig(0.3, 5, n, 0.05, False)), rng


@pytest.mark.parametrize("n", [20000, 400000, 1300000])
def test_chunk_sums_are_bounded(tbem, n):
    _, op, _ = one_leaf(tbem, tbem.LaplaceDouble(), n)
    work = op.info()["work_bytes"]
    print(f"CASE one leaf of {n}: {work / 2**20:.0f} MiB", flush=True)
    assert op.info()["leaf_block"] == 1
    assert work < (2 << 30) + 200 * n


def test_longer_chunks_match_the_direct_sum(tbem):
    torch = pytest.importorskip("torch")
    n, K = 180000, tbem.LaplaceSingle()
    data, op, rng = one_leaf(tbem, K, n)
    print("CASE one leaf, longer chunks", flush=True)
    assert op.info()["work_bytes"] > 1 << 30  # near the bound
    x = torch.tensor(rng.uniform(0.5, 1.5, n), device="cuda")
    ref = tbem.make_direct_nbody_operator(data, K).apply(x).cpu().numpy()
    # one sum of 180,000 positive terms in two orders: a rounding per partial sum
    assert rel_err(op.apply(x).cpu().numpy(), ref) < 1e-12
