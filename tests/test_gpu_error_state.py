"""A HIP call that fails is reported by the call it happened in, and not again by the next
one: after a plan that found no memory the library works as before."""
import importlib

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def test_call_after_an_out_of_memory_error_works(tbem):
    torch = pytest.importorskip("torch")
    error = importlib.import_module("3bem_amd._lib").TbemError
    rng = np.random.default_rng(4)
    n = 150000
    locs, nrm = rng.uniform(0, 1, (n, 3)), rng.standard_normal((n, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    K, w = tbem.LaplaceSingle(), rng.uniform(0.5, 1.5, n)
    make = lambda k, order: tbem.FMMOperator(K, tbem.NBodyData(locs[:k], nrm[:k], locs[:k], nrm[:k], w[:k]),
                                             tbem.FMMConfig(0.3, order, 40, 0.05, False))
    x = torch.tensor(rng.standard_normal(3000), device="cuda")
    y = make(3000, 6).apply(x).cpu().numpy()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    print("CASE out of memory, then a small plan", flush=True)
    # the class operators and output of order 75 take more than 1.5 GiB
    block = torch.empty(torch.cuda.mem_get_info()[0] - (3 << 29), dtype=torch.uint8, device="cuda")
    try:
        with pytest.raises(error, match="memory"):
            make(n, 75)
        z = make(3000, 6).apply(x).cpu().numpy()
    finally:
        del block
        torch.cuda.empty_cache()
    assert rel_err(z, y) < 1e-14
