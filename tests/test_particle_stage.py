"""GPU: the particle stage writes a particle's rows whatever wavefront, lane or launch size it falls in."""
import pytest

import harness as H


def _state(name):
    import geowarp_amd.solvers as gs
    name, _, precision = name.partition(' ')
    cfg = H.MINI[name]()
    if precision:
        cfg['iteration_dict'] = dict(cfg['iteration_dict'], precision=precision)
    s = H.make(gs, cfg)
    total = cfg['total_steps']
    if s.dim == 3:
        s.line_search = True
    s.advance_one_step(0, total)  # a deformed state
    s.prepare_step(1, total)
    return s, s._args(1, total)


@pytest.mark.gpu
@pytest.mark.parametrize('name', ['bar_hencky', 'bar_j2', 'bar_j2 mixed', 'bar_dp', 'bar_norsand', 'terzaghi',
                                  'terzaghi mixed', 'indent_nh', 'indent_nh mixed', 'indent_dp', 'indent_dp mixed'])
def test_stage_rows_do_not_depend_on_the_launch(name):
    """The first k bin-sorted particles of a launch of k (one, a wavefront's and a block's edges) give the
    bits of the launch of all, and nothing behind them is written; without the tangent Y and the states
    are the same and D is left alone."""
    import torch
    s, args = _state(name)
    eng = s.engine
    n, NY, NZ = args.n_particles, eng.NY, eng.NZ
    dev = eng.dev
    arrays = {}
    for k in ('F_new', 'b_new', 'sigma'):
        arrays[k] = torch.empty(n, 9, dtype=torch.float64, device=dev)
        setattr(args, k, arrays[k].data_ptr())
    order = eng.sorted[:n].long()

    def run(k, tangent=True):
        args.n_particles = k
        for a in list(arrays.values()) + [eng.Y, eng.D]:
            a.fill_(float('nan'))
        eng.stage(args, want_tangent=tangent)
        torch.cuda.synchronize()
        out = {q: a[order].clone() for q, a in arrays.items()}
        return dict(out, Y=eng.Y[:n * NY].reshape(n, NY).clone(), D=eng.D[:n * NY * NZ].reshape(n, NY * NZ).clone())

    same = lambda a, b: torch.equal(torch.nan_to_num(a, nan=1e300), torch.nan_to_num(b, nan=1e300))  # noqa: E731
    full = run(n)
    assert not any(bool(torch.isnan(v).any()) for v in full.values())
    for k in (1, 63, 64, 65, 127, 128, 129):
        if k >= n:
            continue
        part = run(k)
        for q, v in part.items():
            assert same(v[:k], full[q][:k]), (k, q)
            assert bool(torch.isnan(v[k:]).all()), (k, q)
    plain = run(n, tangent=False)
    for q, v in plain.items():
        assert bool(torch.isnan(v).all()) if q == 'D' else same(v, full[q]), q
    print(name, 'particles', n, 'max |D|', float(full['D'].abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize('name', ['bar_hencky', 'terzaghi', 'indent_nh'])
def test_g2p_of_any_particle_count(name):
    """G2P of the first n particles (one, a block's edges): the states are copied, the positions are those
    of the launch of all, and nothing behind the n rows is touched."""
    import torch
    s, _ = _state(name)
    eng = s.engine
    N, dim = s.x_particles.shape
    gen = torch.Generator(device=s.device).manual_seed(5)
    rnd = lambda *sh: torch.rand(sh, generator=gen, dtype=torch.float64, device=s.device)  # noqa: E731
    new, old = 1e-3 * rnd(eng.n_nodes * eng.nb), 1e-3 * rnd(eng.n_nodes * eng.nb)
    F, b, al = rnd(N, 9), rnd(N, 9), rnd(N)

    def run(n):
        x, lp = s.x_particles.clone(), s.GIMP_lp.clone()
        Fo, bo, ao, pp = (torch.full(sh, -7.0, dtype=torch.float64, device=s.device) for sh in ((N, 9), (N, 9), (N,), (N,)))
        eng.g2p(x[:n], lp, new, old, Fo, F, bo, b, ao, al, pp)
        torch.cuda.synchronize()
        return x, Fo, bo, ao, pp

    full = run(N)
    assert torch.equal(full[1], F) and torch.equal(full[2], b) and torch.equal(full[3], al)
    assert not torch.equal(full[0], s.x_particles)
    start = (s.x_particles,) + tuple(torch.full_like(a, -7.0) for a in full[1:])
    for n in (1, 127, 128, 129):
        if n >= N:
            continue
        for got, want, before in zip(run(n), full, start):
            assert torch.equal(got[:n], want[:n]) and torch.equal(got[n:], before[n:]), n
