"""A source tree of more cells than one launch's 65,536 tiles of 64 hold (the level products
over every cell): mixed precision, against the direct sum."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def test_products_over_more_tiles_than_a_launch_holds(tbem):
    torch = pytest.importorskip("torch")
    # one point in each cell of a 128^3 grid, eight in the first 260,000 of them: with one
    # point a leaf 3.9 million leaves (fewer than 65,536 tiles) in 4.5 million cells (more)
    grid = (np.stack(np.meshgrid(*[np.arange(128)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) / 128
    half = np.stack(np.meshgrid(*[[-0.25, 0.25]] * 3, indexing="ij"), -1).reshape(-1, 3) / 128
    rng = np.random.default_rng(2)
    grid = grid[rng.permutation(len(grid))]
    src = np.vstack([(grid[:260000, None] + half[None]).reshape(-1, 3), grid[260000:]])
    # observation points close together, so that their cells are small enough for M2L, in the
    # corner whose cells come last
    obs = np.array([[0.97, 0.98, 0.96], [0.9705, 0.98, 0.96], [0.97, 0.9803, 0.96]])
    nrm = lambda m: np.tile([0.0, 0.0, 1.0], (m, 1))
    data, K = tbem.NBodyData(obs, nrm(3), src, nrm(len(src)), np.ones(len(src))), tbem.LaplaceSingle()
    op = tbem.FMMOperator(K, data, tbem.FMMConfig(0.3, 50, 1, 0.05, False), precision="mixed")
    info = op.info()
    print(f"CASE many cells: {info['n_src_cells']} cells, {info['p2m']} leaves, {info['m2l']} M2L pairs, "
          f"plan {info['plan_seconds']:.1f} s", flush=True)
    assert info["n_src_cells"] > 65536 * 64 >= info["p2m"] and info["m2l_classes"] > 0
    x = torch.tensor(rng.uniform(0.5, 1.5, len(src)), device="cuda")
    y = op.apply(x).cpu().numpy()
    assert rel_err(y, tbem.make_direct_nbody_operator(data, K).apply(x).cpu().numpy()) < 1e-5
