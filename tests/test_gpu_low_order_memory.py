"""A low-order plan (below 48 operator rows) on a device with little memory left: the class
M2L, whose operators and per-pair output take gigabytes, gives way to the surfaces, which
need none, instead of failing the plan."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("share", [0.5, 1.5])
def test_low_order_plan_without_room_runs_on_surfaces(tbem, share):
    torch = pytest.importorskip("torch")
    n = 150000
    rng = np.random.default_rng(8)
    locs, nrm = rng.uniform(0, 1, (n, 3)), rng.standard_normal((n, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    K, data = tbem.LaplaceSingle(), tbem.NBodyData(locs, nrm, locs, nrm, rng.uniform(0.5, 1.5, n))
    make = lambda **kw: tbem.FMMOperator(K, data, tbem.FMMConfig(0.3, 44, 40, 0.05, False), **kw)
    free = lambda: (torch.cuda.synchronize(), torch.cuda.empty_cache(), torch.cuda.mem_get_info()[0])[2]
    x = torch.tensor(rng.standard_normal(n), device="cuda")
    roomy = make()
    y = roomy.apply(x).cpu().numpy()
    out = int(roomy.info()["m2l_output_bytes"])
    assert roomy.info()["n_e"] < 48 and roomy.info()["m2l_classes"] > 0 and out > 1e9
    del roomy
    make(translations="surfaces").apply(x)  # (what the runtime keeps after a first use is taken by now)
    before = free()
    surf = make(translations="surfaces")
    held = before - free()
    del surf
    # room for the surfaces' plan and `share` of the class output
    keep = 2 * held + int(share * out)
    print(f"CASE low-order memory: output {out >> 20} MiB, surfaces' plan {held >> 20} MiB, left {keep >> 20} MiB", flush=True)
    assert free() > keep
    block = torch.empty(free() - keep, dtype=torch.uint8, device="cuda")
    try:
        op = make()
        info, z = op.info(), op.apply(x).cpu().numpy()
    finally:
        del block
        torch.cuda.empty_cache()
    assert info["m2l_classes"] == 0 and info["m2l_output_bytes"] == 0
    assert rel_err(z, y) < 1e-9  # the C2E's amplification of last-bit differences, as with room
