"""GPU: particles are ordered by base node, then id, whatever order the atomics of the count give them."""
import numpy as np
import pytest

import oracle.gimp as og


# one particle, empty bins, a block of 256 and its edges, bins of several hundred particles
@pytest.mark.gpu
@pytest.mark.parametrize('cells,n,crowd', [((3, 3), 1, 0), ((4, 5), 255, 0), ((4, 5), 257, 200), ((3, 3, 3), 256, 0),
                                           ((6, 5, 4), 3001, 700), ((30, 20), 5000, 0)])
def test_bins_hold_their_particles_in_order(cells, n, crowd):
    import torch
    from geowarp_amd.solvers._engine import Engine
    dim = len(cells)
    rng = np.random.default_rng(n)
    lp = rng.uniform(0.05, 0.2, (n, dim))
    x = rng.uniform(0, 1, (n, dim)) * np.array(cells) * 0.5
    x[rng.permutation(n)[:crowd]] = 0.6 + 0.01 * rng.random((crowd, dim))
    x = np.clip(x, lp + 1e-3, np.array(cells) * 0.5 - lp - 1e-3)
    eng = Engine(dim, dim == 3, cells, (0.5,) * dim)
    X, LP = (torch.as_tensor(np.ascontiguousarray(a), device=eng.dev) for a in (x, lp))
    lo, ext = zip(*[(lambda r: (r[0], r[4]))(og.axis_weights(x[:, a], lp[:, a], 0.5, 2.0)) for a in range(dim)])
    base = lo[0] + lo[1] * (cells[0] + 1) + (lo[2] * (cells[0] + 1) * (cells[1] + 1) if dim == 3 else 0)
    want = np.lexsort((np.arange(n), base))
    for _ in range(2):  # the second call finds the buffers used
        eng.begin_step(X, LP)
        assert np.array_equal(eng.sorted[:n].cpu().numpy(), want)
        start = eng.cell_start.cpu().numpy()
        assert np.array_equal(np.diff(start), np.bincount(base, minlength=eng.n_nodes))
        assert np.array_equal(eng.x_s[:n * dim].reshape(n, dim).cpu().numpy(), x[want])
        assert np.array_equal(eng.lp_s[:n * dim].reshape(n, dim).cpu().numpy(), lp[want])
        e = sum((np.array(ext[a]) == 3).astype(np.uint8) << a for a in range(dim))
        assert np.array_equal(eng.ext_s[:n].cpu().numpy(), e[want])
