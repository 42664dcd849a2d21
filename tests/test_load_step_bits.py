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


def _engine(cells, n, seed, crowd=0):
    """An engine with random particles on a grid of half-unit cells, `crowd` of them in one cell."""
    import torch
    from geowarp_amd.solvers._engine import Engine
    rng = np.random.default_rng(seed)
    lp = rng.uniform(0.05, 0.25, (n, 3))
    x = rng.uniform(0, 1, (n, 3)) * np.array(cells) * 0.5
    x[:crowd] = 0.6 + 0.02 * rng.random((crowd, 3))
    x = np.clip(x, lp + 1e-3, np.array(cells) * 0.5 - lp - 1e-3)
    eng = Engine(3, True, cells, (0.5, 0.5, 0.5))
    X, LP = (torch.as_tensor(np.ascontiguousarray(a), device=eng.dev) for a in (x, lp))
    eng.begin_step(X, LP)
    return eng, X, LP, rng


def _binned(eng, D, fp32, vals_fp32=False):
    """Binned Jacobian for tangent rows D (bin order), the workspace full of NaN before."""
    import torch
    from geowarp_amd import _lib as L
    from geowarp_amd.solvers._engine import _stream
    lib = L.lib()
    g, b, pat = L.ctypes.byref(eng.grid), L.ctypes.byref(eng.bins), L.ctypes.byref(eng.pattern)
    need = int(lib.gm_node_jacobian_work_bytes(g, int(fp32)))
    w = torch.full((need,), 255, dtype=torch.uint8, device=eng.dev)
    vals = torch.full((eng.nnzb * 16,), float('nan'), dtype=torch.float32 if vals_fp32 else torch.float64,
                      device=eng.dev)
    L.check(lib.gm_node_jacobian_binned(g, b, pat, L.ptr(D), int(fp32), L.ptr(eng.freem), L.ptr(vals),
                                        int(vals_fp32), L.ptr(w), need, _stream()), 'gm_node_jacobian_binned')
    return vals


@pytest.mark.gpu
@pytest.mark.parametrize('cells,n,crowd', [((3, 4, 5), 300, 40), ((20, 5, 4), 3000, 0), ((70, 3, 3), 5000, 30)])
def test_fp32_jacobian_adds_the_bin_sums_in_fp64(cells, n, crowd):
    """The mixed form's matrix adds FP32 sums over a bin's particles in FP64: assembled from the bins of
    even x and from those of odd x (the other particles' tangent zero) the two add up to the whole, to
    the round-off of 27 FP64 additions."""
    import torch
    eng, X, LP, rng = _engine(cells, n, n, crowd)
    eng.freem.fill_(1)
    D = torch.as_tensor(rng.standard_normal((n, 255)).astype(np.float32), device=eng.dev)
    base = torch.repeat_interleave(torch.arange(eng.n_nodes, device=eng.dev),
                                   (eng.cell_start[1:eng.n_nodes + 1] - eng.cell_start[:eng.n_nodes]).long())
    even = (base % (cells[0] + 1) % 2 == 0).to(torch.float32)[:, None]
    whole, a, b = (_binned(eng, (D * m).contiguous(), True) for m in (torch.ones_like(even), even, 1 - even))
    err = float((whole - (a + b)).abs().max() / whole.abs().max())
    print(cells, n, 'even + odd bins against all', err)
    assert float(a.abs().max()) > 0 and float(b.abs().max()) > 0 and err < 1e-14


@pytest.mark.gpu
@pytest.mark.parametrize('cells,n', [((30, 20, 14), 23999), ((30, 20, 14), 24000), ((24, 19, 13), 25000),
                                     ((9, 70, 11), 24100), ((130, 8, 6), 30000)])
def test_fp64_jacobian_either_side_of_the_line_sums(cells, n):
    """The binned FP64 matrix equals the node-row one to the round-off of a differently ordered sum: with
    the particles or the nodes just too few for the line sums, and with enough (lines of one segment and
    of several); all variants write the same bits and every entry."""
    import torch
    from geowarp_amd import _lib as L
    from geowarp_amd.solvers._engine import _stream
    eng, X, LP, rng = _engine(cells, n, 1, 200)
    eng.freem.copy_(torch.as_tensor((rng.random(eng.n_nodes * 4) < 0.9).astype(np.uint8), device=eng.dev))
    D = torch.as_tensor(rng.standard_normal((n, 255)), device=eng.dev)
    b = _binned(eng, D, False)
    lib = L.lib()
    g, bn, pat = L.ctypes.byref(eng.grid), L.ctypes.byref(eng.bins), L.ctypes.byref(eng.pattern)
    a = torch.empty_like(b)
    L.check(lib.gm_node_jacobian(g, bn, pat, L.ptr(D), 0, L.ptr(eng.freem), L.ptr(a), 0, 1, _stream()), 'rows')
    rel = float((a - b).norm() / a.norm())
    print(cells, n, 'nodes', eng.n_nodes, 'bins against rows', rel)
    assert rel < 1e-13  # a few hundred terms of 1e-16
    need = int(lib.gm_node_jacobian_work_bytes(g, 0))
    w, vals = torch.empty(need, dtype=torch.uint8, device=eng.dev), torch.empty_like(b)
    for v in range(4):
        w.fill_(255)
        vals.fill_(float('nan'))
        L.check(lib.gm_jacobian_bins_variant(g, bn, L.ptr(D), 0, v, L.ptr(w), need, _stream()), 'bins')
        L.check(lib.gm_jacobian_gather_variant(g, bn, pat, 0, v % 3, L.ptr(w), L.ptr(eng.freem), L.ptr(vals), 0,
                                               _stream()), 'gather')
        assert torch.equal(vals, b), v


def _sum_by_bins(eng, terms, nb, add=lambda acc, t: acc + t):
    """Nodal sums of per-particle terms (bin order, n x n_nodes x nb): over a bin's particles in their
    order, then over the bins that hold a node in the order of its place in them (x fastest)."""
    nx1, ny1 = eng.grid.nx + 1, eng.grid.ny + 1
    start = eng.cell_start.cpu().numpy()
    bins = np.zeros((eng.n_nodes, eng.n_nodes, nb))
    for b in range(eng.n_nodes):
        for k in range(start[b], start[b + 1]):
            bins[b] = add(bins[b], terms[k])
    i = np.arange(eng.n_nodes)
    c = np.stack([i % nx1, i // nx1 % ny1, i // (nx1 * ny1)], 1)
    out = np.zeros((eng.n_nodes, nb))
    for o in range(27):
        d = np.array([o % 3, o // 3 % 3, o // 9])
        on = (c >= d).all(1)
        out[on] += bins[i[on] - d @ np.array([1, nx1, nx1 * ny1]), i[on]]
    return out


@pytest.mark.gpu
@pytest.mark.parametrize('cells,n,crowd', [((3, 3, 3), 1, 0), ((3, 4, 5), 70, 35), ((5, 2, 3), 90, 0)])
def test_binned_residual_adds_particles_in_bin_order(cells, n, crowd):
    """The residual of all particles is the sum, in bin order, of what each of them gives alone (its row of Y
    the only one that is not zero), bit for bit."""
    import torch
    eng, X, LP, rng = _engine(cells, n, n + 1, crowd)
    eng.freem.fill_(1)
    Y = torch.as_tensor(rng.standard_normal((n, eng.NY)), device=eng.dev)

    def residual(rows):
        eng.Y.view(-1)[:n * eng.NY].copy_(rows.reshape(-1))
        eng._bins_workspace(1 << 20).fill_(255)
        eng.residual(X, LP)
        return eng.rhs.cpu().numpy().reshape(eng.n_nodes, 4).copy()

    one = torch.zeros_like(Y)
    terms = []
    for k in range(n):
        one.zero_()
        one[k] = Y[k]
        terms.append(residual(one))
    assert np.array_equal(residual(Y), _sum_by_bins(eng, terms, 4))


@pytest.mark.gpu
@pytest.mark.parametrize('cells,n,crowd', [((3, 3, 3), 1, 0), ((3, 4, 5), 70, 35), ((5, 2, 3), 90, 0)])
def test_binned_p2g_adds_particles_in_bin_order(cells, n, crowd):
    """The mass projection's right-hand side: w_I m sum_J w_J (a particle alone, of unit pressure) times the
    particle's pressure, added with one rounding, in bin order, then the bins in theirs; bit for bit."""
    from fractions import Fraction
    import torch
    eng, X, LP, rng = _engine(cells, n, n + 2, crowd)
    order = eng.sorted[:n].long()
    p = torch.as_tensor(rng.standard_normal(n), device=eng.dev)

    def rhs(pp):
        eng._bins_workspace(1 << 20).fill_(255)
        return eng.p2g(X, LP, 0.0, None, 0.5, 0.37, pp, mass=True).cpu().numpy().copy()

    one = torch.zeros_like(p)
    terms = []
    for k in range(n):
        one.zero_()
        one[order[k]] = 1.0
        terms.append((rhs(one)[:, None], float(p[order[k]])))
    fma = np.vectorize(lambda a, b, c: float(Fraction(a) * Fraction(b) + Fraction(c)) if a else c)
    assert np.array_equal(rhs(p), _sum_by_bins(eng, terms, 1, lambda acc, t: fma(t[0], t[1], acc))[:, 0])


@pytest.mark.gpu
@pytest.mark.parametrize('cells,n,crowd', [((3, 3, 3), 1, 0), ((3, 4, 4), 50, 40), ((4, 2, 3), 60, 0)])
def test_binned_mass_adds_particles_in_bin_order(cells, n, crowd):
    """The consistent mass (particle mass a power of two) is the sum, in bin order and then over the bins in
    theirs, of what each particle gives alone, bit for bit."""
    import torch
    from geowarp_amd import _lib
    from geowarp_amd.solvers._engine import Engine, _stream
    eng, X, LP, rng = _engine(cells, n, n + 3, crowd)

    def mass(e, x, lp):
        if e.mvals is not None:
            e.mvals.fill_(float('nan'))
        e._bins_workspace(1 << 20).fill_(255)
        e.p2g(x, lp, 0.0, None, 0.5, 0.5, torch.zeros(len(x), dtype=torch.float64, device=e.dev), mass=True)
        rp, ci = e.row_ptr[:e.n_nodes + 1].cpu().numpy(), e.col_idx[:e.nnzb].cpu().numpy()
        M = np.zeros((e.n_nodes, e.n_nodes))
        M[np.repeat(np.arange(e.n_nodes), np.diff(rp)), ci] = e.mvals[:e.nnzb].cpu().numpy()
        return M

    terms = []
    for k in eng.sorted[:n].tolist():
        one = Engine(3, True, cells, (0.5, 0.5, 0.5))
        one.begin_step(X[k:k + 1].contiguous(), LP[k:k + 1].contiguous())
        terms.append(mass(one, X[k:k + 1].contiguous(), LP[k:k + 1].contiguous()))
    assert np.array_equal(mass(eng, X, LP), _sum_by_bins(eng, terms, eng.n_nodes))
    # gm_p2g's own mass (strips of rows) sums the same terms in another order
    L, lib = _lib, _lib.lib()
    vals = torch.full_like(eng.mvals[:eng.nnzb], float('nan'))
    L.check(lib.gm_p2g(L.ctypes.byref(eng.grid), L.ctypes.byref(eng.bins), L.ctypes.byref(eng.pattern), 0.0, None, 0.5,
                       0.5, None, L.ptr(eng.act), L.ptr(eng.bflag), L.ptr(vals), None, _stream()), 'gm_p2g')
    err = float((vals - eng.mvals[:eng.nnzb]).abs().max() / vals.abs().max())
    assert err < 1e-14, err


@pytest.mark.gpu
@pytest.mark.parametrize('options', [0, 3])
@pytest.mark.parametrize('cells', [(2, 3, 2), (4, 4, 4), (13, 9, 11), (41, 30, 28)])
def test_mass_cg_sums_as_the_general_cg(cells, options):
    """gm_pcg_window in 3D, which takes the columns of complete rows from the grid, gives the bits of gm_pcg."""
    import torch
    from geowarp_amd import _lib as L
    from geowarp_amd.solvers._engine import _stream
    eng, X, LP, rng = _engine(cells, 8 * int(np.prod(cells)), 5)
    n, lib = eng.n_nodes, L.lib()
    p = torch.as_tensor(rng.standard_normal(len(X)), device=eng.dev)
    b = eng.p2g(X, LP, 0.0, None, 0.5, 0.7, p, mass=True)
    L.check(lib.gm_fix_empty_diag(n, L.ptr(eng.row_ptr), L.ptr(eng.col_idx), L.ptr(eng.mvals), L.ptr(b), _stream()),
            'gm_fix_empty_diag')
    ws, out = eng.workspace(1, False), []
    for window in (False, True):
        it, rr, x = L.c_int(0), L.c_double(0.0), torch.full_like(b, 0.1)
        tail = (L.ptr(eng.mvals), L.ptr(b), L.ptr(x), L.ctypes.byref(ws), 1e-10, 4000, 16, options,
                L.ctypes.byref(it), L.ctypes.byref(rr), _stream())
        if window:
            L.check(lib.gm_pcg_window(L.ctypes.byref(eng.grid), L.ctypes.byref(eng.pattern), *tail), 'window')
        else:
            L.check(lib.gm_pcg(1, 0, n, L.ptr(eng.row_ptr), L.ptr(eng.col_idx), *tail), 'general')
        out.append((x, it.value, rr.value))
    print(cells, options, out[0][1:], out[1][1:])
    assert torch.equal(out[0][0], out[1][0]) and out[0][1:] == out[1][1:]


def _tree(v):
    """Sum over the last axis, 256 long, halves added onto each other."""
    while v.shape[-1] > 1:
        v = v[..., :v.shape[-1] // 2] + v[..., v.shape[-1] // 2:]
    return v[..., 0]


def _dot(a, b, chunks):
    """Sum of FP32 products in FP64: chunks of 256 threads in turn, a tree over each chunk's threads, then
    256 threads over the chunks and a tree."""
    def strided(v, width):
        v = np.pad(v, (0, -len(v) % width)).reshape(-1, width)
        s = np.zeros(width)
        for row in v:
            s = s + row
        return s
    part = _tree(strided(a.astype(np.float64) * b.astype(np.float64), chunks * 256).reshape(chunks, 256))
    return _tree(strided(part, 256))


@pytest.mark.gpu
@pytest.mark.parametrize('n', [65537, 131072, 300001])
@pytest.mark.parametrize('near', [False, True])
def test_gmres_sums_of_long_vectors(n, near):
    """One step of FP32 GMRES on a system of more than 65,536 unknowns: its residual estimate from sums in
    the stated order (products with a basis vector in 256 chunks, norms in up to 1024, that of a second
    pass in 256), bit for bit.  near: the first pass removes almost all of w and a second one follows."""
    import torch
    from geowarp_amd import _lib as L
    from geowarp_amd.solvers._engine import _stream
    rng = np.random.default_rng(n)
    f32 = np.float32
    lower, upper = ((rng.random(n) * (1e-3 if near else 3.0)).astype(f32) for _ in range(2))
    lower[0] = upper[-1] = 0.0
    diag = np.where(rng.random(n) < 0.5, f32(1), f32(2))  # (its inverse is exact)
    b = rng.standard_normal(n).astype(f32)
    i = np.arange(n)
    cols = np.stack([i - 1, i, i + 1], 1)
    ok = (cols >= 0) & (cols < n)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device='cuda')  # noqa: E731
    rp, ci = t(np.r_[0, ok.sum(1).cumsum()].astype(np.int32)), t(cols[ok].astype(np.int32))
    vals, B = t(np.stack([lower, diag, upper], 1)[ok]), t(b)
    m = 12
    x, z, w, dinv = (torch.zeros(n, dtype=torch.float32, device='cuda') for _ in range(4))
    V = torch.zeros(m + 1, n, dtype=torch.float32, device='cuda')
    part = torch.zeros(2048, dtype=torch.float64, device='cuda')
    dh = torch.zeros(3 * (m + 2), dtype=torch.float64, device='cuda')
    its, rel = L.c_int(0), L.c_double(0.0)
    L.check(L.lib().gm_gmres(1, 1, n, L.ptr(rp), L.ptr(ci), L.ptr(vals), L.ptr(B), L.ptr(x), L.ptr(V), L.ptr(z),
                             L.ptr(w), L.ptr(dinv), L.ptr(part), L.ptr(dh), m, 1e-12, 1, L.ctypes.byref(its),
                             L.ctypes.byref(rel), _stream()), 'gm_gmres')
    f64 = lambda a: a.astype(np.float64)  # noqa: E731
    nv = min(1024, -(-n // 256))  # chunks of a norm
    beta = np.sqrt(_dot(b, b, nv))
    v = (f64(b) * (1.0 / beta)).astype(f32)
    y = f64(v / diag)
    q = np.r_[0.0, y, 0.0]
    u = (f64(lower) * q[:-2] + f64(diag) * y + f64(upper) * q[2:]).astype(f32)
    h, before = _dot(v, u, 256), _dot(u, u, nv)
    u = (f64(u) - h * f64(v)).astype(f32)
    after = _dot(u, u, nv)
    assert (after < 0.5 * before) == near
    if near:
        h2 = _dot(v, u, 256)
        u = (f64(u) - h2 * f64(v)).astype(f32)
        h, after = h + h2, _dot(u, u, 256)
    hn = np.sqrt(after)
    want = abs(-(hn / np.sqrt(h * h + hn * hn)) * beta) / beta
    print(n, near, rel.value, want)
    assert its.value == 1 and rel.value == want


@pytest.mark.gpu
def test_mixed_3d_hierarchy_keeps_the_host_inverse():
    """The coarsest operator of the 3D mixed form's hierarchy, which is kept across load steps, is inverted by
    LU on the host, bit for bit."""
    from test_dense_inverse import _coarsest, _solved
    from geowarp_amd.solvers import _multigrid as MG
    s, mgh = _solved('indent', 'mixed')
    A = _coarsest(mgh)
    assert mgh.dense and mgh.fp32
    assert np.array_equal(mgh.cinv.cpu().numpy().reshape(A.shape), MG._robust_inverse(A))


@pytest.mark.gpu
@pytest.mark.parametrize('stiffness,depth', [(0.921, 0.044), (0.902, 0.0441), (1.114, 0.0438), (0.992, 0.0438),
                                             (0.946, 0.0509), (0.868, 0.0459)])
def test_large_mixed_load_steps_clip_the_same_domains(stiffness, depth):
    """Three load steps of the 64 x 64 x 32-cell indentation (mixed form): the 16,384 particles of the bottom
    layer whose domains the box cuts are those of the fixture, recorded before the kernels of the step were
    made faster.  On these six paths a sum in another order in any of the stage, the residual, the Jacobian,
    the P2G, the mass or the coarsest inverse flips one to twenty of them."""
    import os
    import geowarp_amd.solvers as gs
    from geowarp_amd import problems as P
    cfg = P.indent3d(material='Neo-Hookean', precision='mixed', tol=1e-10, n_iter=12, footing=0.2, depth=depth,
                     footing_start='surface', penalty_form='physical', dp_apex='return', shape_factor=0.1)
    cfg['material_dict']['youngs_modulus'] *= stiffness
    s = P.build_solver(gs, cfg, device='cuda')
    cfg['particle_flags'](s.x_particles, s.particle_traction_flag_array, s.particle_pressure_boundary_flag_array)
    s.line_search = True
    s.linear_maxiter = 1500
    bottom = s.x_particles[:, 2] < 0.5 * s.dz
    for k in range(3):
        s.advance_one_step(k, cfg['total_steps'])
    cut = (s.GIMP_lp[:, 2] == s.x_particles[:, 2] - s.domain_min_z - 1e-6)[bottom].cpu().numpy()
    with np.load(os.path.join(os.path.dirname(__file__), 'golden', 'indent_mixed_clips.npz')) as f:
        want = np.unpackbits(f['%s_%s' % (stiffness, depth)]).astype(bool)
    print(stiffness, depth, 'cut', int(cut.sum()), 'of', cut.size, 'other', int((cut != want).sum()))
    assert cut.size == want.size == 16384
    assert np.array_equal(cut, want)
