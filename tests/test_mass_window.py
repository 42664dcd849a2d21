"""GPU: conjugate gradients on the consistent mass in the grid's pattern (gm_pcg_window) against the
general ones (gm_pcg)."""
import numpy as np
import pytest


def _mass_system(cells, ppd, seed=0):
    """Engine of a 2D or 3D u-p grid with ppd^dim particles a cell at random places, its consistent mass
    and a right-hand side."""
    import torch
    from geowarp_amd.solvers._engine import Engine
    dim = len(cells)
    h = (0.5,) * dim
    rng = np.random.default_rng(seed)
    n = int(np.prod(cells)) * ppd ** dim
    lp = rng.uniform(0.05, 0.25, (n, dim))
    x = rng.uniform(0, 1, (n, dim)) * np.array(cells) * 0.5
    x = np.clip(x, lp + 1e-3, np.array(cells) * 0.5 - lp - 1e-3)
    eng = Engine(dim, True, cells, h)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=eng.dev)  # noqa: E731
    X, LP = t(x), t(lp)
    eng.begin_step(X, LP)
    pbc = torch.zeros(n, dtype=torch.uint8, device=eng.dev)
    mrhs = eng.p2g(X, LP, 1e-9, pbc, 0.0, 0.7, t(rng.standard_normal(n)), mass=True)
    return eng, mrhs, x, lp


# no complete row, or one at most; many; more rows than the 1024 workgroups hold at once
@pytest.mark.gpu
@pytest.mark.parametrize('cells', [(3, 3), (4, 4), (37, 23), (300, 260), (2, 3, 2), (4, 4, 4), (13, 9, 11),
                                   (40, 31, 29)])
@pytest.mark.parametrize('options', [0, 3])
def test_window_cg_equals_general_cg(cells, options):
    import torch
    from geowarp_amd import _lib as L
    from geowarp_amd.solvers._engine import _stream
    eng, b, _, _ = _mass_system(cells, 3)
    lib = L.lib()
    n = eng.n_nodes
    L.check(lib.gm_fix_empty_diag(n, L.ptr(eng.row_ptr), L.ptr(eng.col_idx), L.ptr(eng.mvals), L.ptr(b), _stream()),
            'gm_fix_empty_diag')
    full = int((eng.row_ptr[1:n + 1] - eng.row_ptr[:n] == 5 ** len(cells)).sum())
    ws = eng.workspace(1, False)
    tol, out = 1e-12, []
    for window in (False, True):
        it, rr = L.c_int(0), L.c_double(0.0)
        x = torch.full_like(b, 0.1)
        tail = (L.ptr(eng.mvals), L.ptr(b), L.ptr(x), L.ctypes.byref(ws), tol, 4000, 16, options, L.ctypes.byref(it),
                L.ctypes.byref(rr), _stream())
        if window:
            L.check(lib.gm_pcg_window(L.ctypes.byref(eng.grid), L.ctypes.byref(eng.pattern), *tail), 'window')
        else:
            L.check(lib.gm_pcg(1, 0, n, L.ptr(eng.row_ptr), L.ptr(eng.col_idx), *tail), 'general')
        r = torch.empty_like(b)
        L.check(lib.gm_bsr_spmv(1, 0, 0, n, L.ptr(eng.row_ptr), L.ptr(eng.col_idx), L.ptr(eng.mvals), L.ptr(x),
                                L.ptr(r), _stream()), 'spmv')
        out.append((x, it.value, rr.value, float((r - b).norm() / b.norm())))
    (x0, i0, r0, t0), (x1, i1, r1, t1) = out
    print(cells, options, 'rows', n, 'complete', full, 'iterations', i0, i1, 'relres', r0, r1, 'true', t0, t1)
    assert full > 0 if min(cells) >= 9 else full <= 1
    # both meet the tolerance; the sums are the same but for their order, so the counts differ by a
    # few of the last iterations at most
    assert r0 <= tol and r1 <= tol and t1 <= 2e-12 and abs(i0 - i1) <= 0.05 * i0 + 2


@pytest.mark.gpu
def test_window_cg_reports_what_the_general_cg_reports():
    """NaN in the right-hand side is refused, zero gives zero, and an indefinite matrix stops the
    iteration on the device."""
    import torch
    from geowarp_amd import _lib as L
    from geowarp_amd.solvers._engine import _stream
    eng, b, _, _ = _mass_system((6, 5, 7), 1)
    lib, n = L.lib(), eng.n_nodes
    ws = eng.workspace(1, False)

    def solve(b, vals):
        it, rr = L.c_int(0), L.c_double(0.0)
        x = torch.full_like(b, 0.1)
        rc = lib.gm_pcg_window(L.ctypes.byref(eng.grid), L.ctypes.byref(eng.pattern), L.ptr(vals), L.ptr(b), L.ptr(x),
                               L.ctypes.byref(ws), 1e-12, 200, 16, 0, L.ctypes.byref(it), L.ctypes.byref(rr),
                               _stream())
        return rc, it.value, rr.value, x

    bad = b.clone()
    bad[n // 2] = float('nan')
    assert solve(bad, eng.mvals)[0] == -5
    rc, its, rel, x = solve(torch.zeros_like(b), eng.mvals)
    assert rc == 0 and its == 0 and float(x.abs().max()) == 0.0
    rc, its, rel, x = solve(b, -eng.mvals)
    assert rc == 0 and its <= 200 and rel > 1e-12


# fewer rows than a strip of 21, remainders, grid lines shorter and longer than a strip, and (crowd) bins
# whose ranges take several pieces of 96 particles
@pytest.mark.gpu
@pytest.mark.parametrize('cells', [(2, 2), (3, 6), (20, 3), (41, 7), (2, 2, 2), (6, 4, 3), (21, 3, 4), (3, 5, 9)])
@pytest.mark.parametrize('crowd', [False, True])
def test_mass_matrix_equals_the_dense_sum(cells, crowd):
    """M_IJ = m sum_p w_I w_J with the oracle's weights, every entry of the pattern written; the
    right-hand side is m sum_p w_I p_p sum_J w_J."""
    import torch
    import oracle.gimp as og
    eng, b, x, lp = _mass_system(cells, 8 if crowd else 2, seed=1)
    dim, N = len(cells), eng.n_nodes
    lo, w, _, _, _ = zip(*[og.axis_weights(x[:, a], lp[:, a], 0.5, 2.0) for a in range(dim)])
    # dense products one axis at a time: W_a (particles x nodes of the axis)
    W = []
    for a in range(dim):
        Wa = np.zeros((len(x), cells[a] + 3))
        for i in range(3):
            np.add.at(Wa, (np.arange(len(x)), lo[a] + i), w[a][:, i])
        W.append(Wa[:, :cells[a] + 1])
    P = W[0]
    for a in range(1, dim):
        P = np.einsum('pi,pj->pij', W[a], P.reshape(len(x), -1)).reshape(len(x), -1)  # x fastest
    M = 0.7 * P.T @ P
    rp, ci = eng.row_ptr[:N + 1].cpu().numpy(), eng.col_idx[:eng.nnzb].cpu().numpy()
    got = np.zeros((N, N))
    got[np.repeat(np.arange(N), np.diff(rp)), ci] = eng.mvals[:eng.nnzb].cpu().numpy()
    err = np.abs(got - M).max() / np.abs(M).max()
    print(cells, crowd, 'particles', len(x), 'entries', eng.nnzb, 'max error', err)
    assert err < 1e-13  # sums of up to a few thousand positive terms of 1e-16 each
    eng.mvals.fill_(float('nan'))
    X, LP = (torch.as_tensor(np.ascontiguousarray(q), device=eng.dev) for q in (x, lp))
    pp = torch.as_tensor(np.random.default_rng(2).standard_normal(len(x)), device=eng.dev)
    b = eng.p2g(X, LP, 1e-9, torch.zeros(len(x), dtype=torch.uint8, device=eng.dev), 0.0, 0.7, pp, mass=True)
    assert not bool(torch.isnan(eng.mvals[:eng.nnzb]).any())
    r = 0.7 * P.T @ (pp.cpu().numpy() * P.sum(1))
    assert np.abs(b.cpu().numpy() - r).max() < 1e-12 * np.abs(r).max()
