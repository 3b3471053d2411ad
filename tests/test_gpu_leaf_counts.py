"""tbem_fmm_info's counts of the leaf stage's work: leaf_chunked counts the leaves that the
one-wave kernel runs in chunks, not those that the one-workgroup kernel cuts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,leaf,wave", [(3000, 4000, False), (20000, 3000, False), (3000, 60, True)])
def test_chunked_leaves_are_the_wave_kernels(tbem, n, leaf, wave):
    rng = np.random.default_rng(n)
    locs, nrm = rng.uniform(0, 1, (n, 3)), rng.standard_normal((n, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    op = tbem.FMMOperator(tbem.LaplaceDouble(), tbem.NBodyData(locs, nrm, locs, nrm, np.ones(n)),
                          tbem.FMMConfig(0.3, 5, leaf, 0.05, False))
    inf = op.info()
    print(f"CASE leaf counts n={n} leaf={leaf}: " + str({k: inf[k] for k in inf if k.startswith("leaf")}), flush=True)
    if wave:
        assert inf["leaf_block"] == 0 and inf["leaf_wave_items"] > 0
    else:
        assert inf["leaf_wave_items"] == 0 and inf["leaf_chunked"] == 0 and inf["leaf_block"] > 0
    assert inf["leaf_chunked"] <= inf["leaf_wave_items"]
