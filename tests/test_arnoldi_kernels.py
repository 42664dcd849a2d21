"""GPU: the Gram-Schmidt kernels of the Arnoldi step over the sizes their launches depend on."""
import numpy as np
import pytest

from geowarp_amd import _lib as L


# fewer entries than a thread block, a chunk of 1024 and its edges, the last size whose products the
# update sums itself and the first it does not, more rows than the update's 1024 blocks hold at once
@pytest.mark.gpu
@pytest.mark.parametrize('fp32', [False, True])
@pytest.mark.parametrize('n', [2, 255, 1025, 16 * 1024 + 1, 65536, 65537, 300001])
@pytest.mark.parametrize('near', [False, True])
def test_arnoldi_basis_is_orthonormal_and_solves(n, fp32, near):
    """A tridiagonal system with block-Jacobi GMRES(m).  near: A M^-1 = I + small, so the first pass
    removes almost all of w and the second decides the basis; otherwise most steps take one pass.
    The basis is orthonormal, the solution meets the tolerance, and the workspace ends where the
    interface says."""
    import torch
    lib = L.lib()
    m = 12
    dt = torch.float32 if fp32 else torch.float64
    gen = torch.Generator(device='cuda').manual_seed(n)
    off = 1e-3 if near else 0.45
    i = torch.arange(n, device='cuda')
    cols = torch.stack([i - 1, i, i + 1], 1)
    ok = (cols >= 0) & (cols < n)
    v = torch.rand((n, 3), generator=gen, device='cuda', dtype=torch.float64) * off
    v[:, 1] = 1.0
    rp = torch.cat([torch.zeros(1, device='cuda', dtype=torch.int64), ok.sum(1).cumsum(0)]).int()
    ci, vals = cols[ok].int(), v[ok].to(dt)
    b = torch.randn(n, generator=gen, device='cuda', dtype=torch.float64).to(dt)
    x, z, w, dinv = (torch.zeros(n, dtype=dt, device='cuda') for _ in range(4))
    V = torch.zeros(m + 1, n, dtype=dt, device='cuda')
    cap, nd = max(64 * (m + 1), 2048), 3 * (m + 2)
    part = torch.full((cap + 8,), 7.0, dtype=torch.float64, device='cuda')
    dh = torch.full((nd + 8,), 7.0, dtype=torch.float64, device='cuda')
    its, rel = L.c_int(0), L.c_double(0.0)
    tol = 1e-4 if fp32 else 1e-7
    L.check(lib.gm_gmres(1, int(fp32), n, L.ptr(rp), L.ptr(ci), L.ptr(vals), L.ptr(b), L.ptr(x), L.ptr(V), L.ptr(z),
                         L.ptr(w), L.ptr(dinv), L.ptr(part), L.ptr(dh), m, tol, 200, L.ctypes.byref(its),
                         L.ctypes.byref(rel), L.c_void_p(torch.cuda.current_stream().cuda_stream)), 'gm_gmres')
    torch.cuda.synchronize()
    xp = torch.cat([torch.zeros(1, device='cuda', dtype=torch.float64), x.double(),
                    torch.zeros(1, device='cuda', dtype=torch.float64)])
    vd = torch.where(ok, v.to(dt).double(), torch.zeros((), device='cuda', dtype=torch.float64))
    r = b.double() - (vd[:, 0] * xp[:-2] + vd[:, 1] * xp[1:-1] + vd[:, 2] * xp[2:])
    true = float(r.norm() / b.double().norm())
    k = (its.value - 1) % m + 1  # vectors of the last cycle, the one after them included if not a breakdown
    Q = V[:min(k, n)].double()
    dev = float((Q @ Q.T - torch.eye(Q.shape[0], device='cuda', dtype=torch.float64)).abs().max())
    print(n, fp32, near, 'iterations', its.value, 'relative residual', true, 'estimate', rel.value, 'V^T V - I', dev)
    assert 1 <= its.value < 200
    # the estimate is the true residual up to the rounding of x and of the products
    assert true <= (2e-4 if fp32 else 1.1e-7)
    # after two passes a few rounding units; one pass that removes at most half leaves about as many a step
    assert dev < (2e-5 if fp32 else 1e-13)
    assert bool((part[cap:] == 7.0).all()) and bool((dh[nd:] == 7.0).all())
