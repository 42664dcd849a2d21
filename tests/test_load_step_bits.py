"""GPU: the order and the rounding of the sums that the load steps of the 3D u-p form depend on.

The end of a load step clips a particle's domain where it sticks out of the particle-domain box
(update_GIMP_lp_3d, gimp.py:489-505): a jump of 1e-6 that hangs, for the particles in the box's wall
cells, on the last digits of their position and deformation gradient.  A sum taken in another order
moves the Newton iterates within their tolerance and flips some of those entries, so the kernels on
the way there keep their sums' order.
"""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize('n', [1, 257, 20000])
def test_gimp_end_gradients_round_like_the_quotients(n):
    """-a / (2 h lp) * d / |d| of the end nodes: a product and two quotients, each rounded (h a power of
    two, so that the node positions are exact)."""
    import torch
    from geowarp_amd import _lib as L
    from geowarp_amd.solvers._engine import _stream
    rng = np.random.default_rng(n)
    h = 1.0 / 64
    lp = rng.uniform(0.1, 0.5, (n, 2)) * h
    x = rng.uniform(3, 9, (n, 2)) * h
    X, LP = (torch.as_tensor(v, device='cuda') for v in (x, lp))
    out = torch.empty(n, 6, 2, dtype=torch.float64, device='cuda')
    L.check(L.lib().gm_gimp_weights(n, 2, L.ptr(X), L.ptr(LP), (L.ctypes.c_double * 2)(h, h), L.ptr(out), None, None,
                                    _stream()), 'gm_gimp_weights')
    g = out.cpu().numpy()[:, 3:]
    lo, hi = (np.trunc((x + s * lp) / h + 1e-8) for s in (-1.0, 1.0))
    wide = lo != hi
    assert wide.any() or n == 1
    for k in (0, 2):
        d = x - (lo + k) * h
        ref = -((h + lp) - np.abs(d)) / (2.0 * h * lp) * d / np.abs(d)
        assert np.array_equal(g[:, k][wide], ref[wide]), k
