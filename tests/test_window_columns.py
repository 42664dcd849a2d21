"""GPU: level products that take a full row's columns from the grid write the bits of those that read them."""
import ctypes

import numpy as np
import pytest


# no full row, one, and grids whose lines and planes differ
@pytest.mark.gpu
@pytest.mark.parametrize('cells', [(2, 3, 2), (4, 4, 4), (9, 5, 6)])
@pytest.mark.parametrize('nb', [3, 4])
@pytest.mark.parametrize('kind', ['fp64', 'fp32', 'fp16'])
def test_full_rows_take_their_columns_from_the_grid(cells, nb, kind):
    import torch
    from geowarp_amd import _lib as L
    from geowarp_amd.solvers._engine import _stream
    from geowarp_amd.solvers._multigrid import window_pattern
    dev = torch.device('cuda')
    gen = torch.Generator(device=dev).manual_seed(nb)
    rp, ci, mask = window_pattern(3, cells)
    # every seventh row without its last block: a partial row inside the grid
    n = len(rp) - 1
    keep = np.ones(len(ci), bool)
    for i in range(0, n, 7):
        keep[rp[i + 1] - 1] = False
        m = mask[i].view(np.uint64).copy()
        w = 1 if m[1] else 0
        m[w] &= ~(np.uint64(1) << np.uint64(int(m[w]).bit_length() - 1))
        mask[i] = m.view(np.int64)
    rp = np.concatenate([[0], np.cumsum(np.add.reduceat(keep, rp[:-1]))]).astype(np.int32)
    ci = ci[keep]
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
    rp_, ci_, mk = t(rp), t(ci), t(mask.reshape(-1))
    dt = torch.float64 if kind == 'fp64' else torch.float32
    rnd = lambda *s: torch.randn(s, generator=gen, device=dev, dtype=torch.float64)  # noqa: E731
    vals, x, b, dinv = rnd(len(ci) * nb * nb).to(dt), rnd(n * nb).to(dt), rnd(n * nb).to(dt), rnd(n * nb * nb).to(dt)
    lo, scale = rnd(len(ci) * nb * nb).half(), rnd(n * nb * nb).float().abs()
    lv = L.gm_mg_level()
    lv.nx, lv.ny, lv.nz = cells
    lv.n_nodes, lv.nnzb = n, len(ci)
    lv.row_ptr, lv.col_idx, lv.vals, lv.dinv = rp_.data_ptr(), ci_.data_ptr(), vals.data_ptr(), dinv.data_ptr()
    if kind == 'fp16':
        lv.vals_lo, lv.row_scale = lo.data_ptr(), scale.data_ptr()
    full = int((np.diff(rp) == 125).sum())
    for mode in (1, 2):
        out = []
        for m in (None, mk.data_ptr()):
            lv.row_mask = m
            o = torch.full_like(x, float('nan'))
            L.check(L.lib().gm_mg_level_op(nb, int(kind != 'fp64'), ctypes.addressof(lv), 0, mode, L.ptr(x), L.ptr(b),
                                           0.4, L.ptr(o), _stream()), 'gm_mg_level_op')
            out.append(o)
        torch.cuda.synchronize()
        print(cells, nb, kind, 'mode', mode, 'full rows', full, 'of', n, float(out[0].abs().max()))
        assert not bool(torch.isnan(out[0]).any()) and torch.equal(out[0], out[1])
    assert full > 0 or min(cells) <= 4
