"""tbem_fmm_stage_times with the point pairs on the second stream: the far field's stages
report their own time, not their wait for the point pairs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# few levels and heavy leaves (one, three and four levels): the point pairs take several times
# the far field's time
@pytest.mark.parametrize("n,leaf", [(8000, 10000), (30000, 4000), (40000, 600)])
def test_far_field_times_leave_out_the_point_pairs(tbem, n, leaf):
    rng = np.random.default_rng(n)
    locs, nrm = rng.uniform(0, 1, (n, 3)), rng.standard_normal((n, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    op = tbem.FMMOperator(tbem.ElasticHypersingular(1.0, 0.25), tbem.NBodyData(locs, nrm, locs, nrm, np.ones(n)),
                          tbem.FMMConfig(0.3, 5, leaf, 0.05, False))
    x = rng.standard_normal(3 * n)
    far = ("gather", "p2m", "m2m", "m2l", "l2l")
    seen = {}
    for on in (False, True):
        op.set_overlap(on)
        op.apply(x)
        best = [op.apply(x) is not None and op.stage_times() for _ in range(3)]
        seen[on] = {k: min(t[k] for t in best) for k in best[0]}
    print(f"CASE stage times n={n} leaf={leaf} levels={op.info()['n_down_levels']}: {seen}", flush=True)
    off, on = seen[False], seen[True]
    assert off["leaf"] > 3 * sum(off[k] for k in far)  # what the case is for
    for t in (off, on):
        assert all(v >= 0 for v in t.values())
        # beside the point pairs the far field's kernels share the chip with them, but a stage
        # that waited for their end would show most of their time
        assert t["m2l"] < 0.5 * off["leaf"] and t["l2l"] < 0.5 * off["leaf"]
