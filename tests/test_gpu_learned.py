"""Transient INS on the channel with holes (implicit Euler + Oseen Picard,
opencmp/models/ins.py:323-359) with the Schur-diagonal preconditioner, and what
the learned initial guess gains over the plain one on the same steps."""
import numpy as np
import pytest
import torch

from opencmp_amd import _lib as L

pytestmark = pytest.mark.gpu


def say(*a):
    print('[gpu-test]', *a, flush=True)


def channel_model(ctx, n, precision='fp64', tol=1e-8):
    from opencmp_amd.mesh import channel_with_holes
    from opencmp_amd.models import INS, const
    hm = channel_with_holes(n)
    inflow = [(L.FN_POLY2, [0, 0, 6.0, 0, 0, -6.0]), const(0.0)]     # u = (4 * 1.5 y (1 - y), 0)
    zero = [const(0.0), const(0.0)]
    return INS(hm, kv=1e-3, interp_ord=2, dirichlet={'u': {'inlet': inflow, 'wall': zero, 'cyl': zero}},
               linear_solver='GMRes', preconditioner='schur', linear_tolerance=tol, restart=100,
               nonlinear_tolerance=(1e-6, 1e-6), nonlinear_max_iters=3, precision=precision, ctx=ctx)


def test_channel_ins_transient_schur(gpu_ctx):
    from opencmp_amd.solvers import ImplicitEulerSolver
    say('channel INS n=24, 4 implicit Euler steps dt 1e-3, GMRES + Schur diagonal')
    m = channel_model(gpu_ctx, 24)
    s = ImplicitEulerSolver(m, dt=1e-3)
    for k in range(4):
        r = s.step()
        say(f'  step {k}: picard {m.picard_iterations} err {m.picard_error:.2e} lin iters {m.linear_iterations} '
            f'res {r.rel_residual:.2e} log {m.picard_log}')
        assert r.converged and r.rel_residual <= 1e-8
    u = s.gfu_prev.vec
    assert torch.isfinite(u).all()
    nu = m.fes.blocks[0][1]
    say('  max |u_x|', float(u[:nu].abs().max()), 'max |p|', float(u[2 * nu:].abs().max()))


def test_guess_choice_on_the_device_matches_the_host_rule(gpu_ctx):
    """choose_best_async (residuals, choice and copy of the winner all on the device, the outcome read
    afterwards) against choose_best (residuals read back, choice on the host) on the same system:
    a NaN candidate never wins, the first of two equal best candidates wins, a worse candidate loses
    to the plain guess, and a NaN plain residual keeps the plain guess."""
    from opencmp_amd.learned import choose_best, choose_best_async
    from opencmp_amd.solvers import ImplicitEulerSolver
    say('guess choice: device rule against the host rule')
    m = channel_model(gpu_ctx, 16)
    s = ImplicitEulerSolver(m, dt=1e-3)
    for _ in range(2):
        s.step()
    a, b = s.a, s.L.vec
    x0 = s.gfu_prev.vec.clone()  # solves the last Picard system, the one `a` holds
    g = torch.Generator(device=x0.device).manual_seed(3)
    worse = x0 + 1e-3 * torch.randn(x0.shape, generator=g, device=x0.device, dtype=x0.dtype)
    nan = x0.clone()
    nan[5] = float('nan')
    cases = [(worse, [('nan', nan), ('good', x0), ('dup', x0.clone())], 'good'),
             (x0, [('worse', worse)], 'plain'),
             (nan, [('good', x0)], 'plain')]
    for plain, cands, expect in cases:
        p_host, p_dev = plain.clone(), plain.clone()
        host = choose_best(a, b, p_host, cands)
        dev = choose_best_async(a, b, p_dev, cands)()
        say('  host', host, 'device', dev)
        assert host[0] == dev[0] == expect
        assert (host[1] == dev[1] or (np.isnan(host[1]) and np.isnan(dev[1]))) and host[2] == dev[2]
        assert torch.equal(p_host.view(torch.int64), p_dev.view(torch.int64))


def test_learned_guess_lowers_picard_error_at_equal_work(gpu_ctx):
    """Train the MLP on 40 plain steps, then run 8 more steps from the same state with the plain
    and with the learned guess. Measured gain: the learned guess wins the residual comparison on
    every step it is chosen and leaves the truncated Picard iteration closer to its fixed point
    (lower final Picard error); it does not save linear iterations (within 10 %), which this test
    states rather than claims a reduction."""
    from opencmp_amd.learned import GuessPolicy, MLPGuess
    from opencmp_amd.solvers import ImplicitEulerSolver
    say('learned guess: 40 recorded steps, train, 8 compared steps')
    m = channel_model(gpu_ctx, 24)
    n = m.fes.ndof
    pol = GuessPolicy(gpu_ctx, n, max_snapshots=64)
    s = ImplicitEulerSolver(m, dt=1e-3, guess=pol)
    for _ in range(40):
        s.step()
    state = s.gfu_prev.vec.clone()
    ring = [h.clone() for h in pol.history()]
    snap = pol.snapshots()
    say('  snapshots', tuple(snap.shape), 'norms', [round(float(v), 4) for v in snap.norm(dim=1)[::8]])
    net = MLPGuess(gpu_ctx, seed=0, max_batch=16384)
    # the network predicts the velocity blocks; the pressure (a Lagrange multiplier) keeps the plain guess
    nvel = len(m.fes.comp_blocks[0])
    seg = [int(v) for v in m.fes.block_offsets()[:nvel + 1]]
    losses = net.train(snap, seg, steps=600, batch=16384, lr=2e-3, seed=1)
    X, T = net.sample(snap, seg[-1], 7, 4096)
    say('  scales', net.scales(), 'X rms', X.pow(2).mean(0).sqrt().tolist(), 'T rms', float(T.pow(2).mean().sqrt()))
    say('  loss', losses[0], '->', losses[-1])
    assert losses[-1] < 0.2 * losses[0]

    def run(use_net):
        mm = channel_model(gpu_ctx, 24)
        p2 = GuessPolicy(gpu_ctx, n, net=net if use_net else None, n_learned=seg[-1])
        for h in reversed(ring[1:]):  # u^{n-3}, u^{n-2}, u^{n-1}; the solver pushes u^n itself
            p2.push(h)
        g0 = type(s.gfu_prev)(mm.fes, state.clone())
        # the chosen guess is also the first Picard linearisation point
        ss = ImplicitEulerSolver(mm, dt=1e-3, gfu0=g0, guess=p2, linearize_at_guess=True)
        mm.W.vec.copy_(state)
        its, pic, perr = 0, 0, []
        for _ in range(8):
            ss.step()
            its += mm.linear_iterations
            pic += mm.picard_iterations
            perr.append(mm.picard_error)
            say('   ', 'learned' if use_net else 'plain', mm.picard_log)
        return ss.gfu_prev.vec.clone(), its, pic, ss.guess_log, perr

    u_plain, it_plain, pic_plain, _, perr_plain = run(False)
    u_learn, it_learn, pic_learn, log, perr_learn = run(True)
    say(f'  plain: {it_plain} iters / {pic_plain} picard; learned: {it_learn} iters / {pic_learn} picard')
    say('  choices', [c for c, _, _ in log])
    say('  final Picard errors plain', perr_plain, 'learned', perr_learn)
    assert all(rl < rp for c, rp, rl in log if c == 'learned')
    assert sum(c == 'learned' for c, _, _ in log) >= 5
    # the learned guess puts the Oseen iterate closer to the fixed point at no extra linear work
    assert np.mean(perr_learn) < 0.8 * np.mean(perr_plain)
    assert it_learn <= 1.1 * it_plain
    # both runs are the same discretisation; they differ by the truncated Picard iteration only
    rel = float(torch.linalg.norm(u_learn - u_plain) / torch.linalg.norm(u_plain))
    say('  rel diff of the final states', rel)
    assert rel < 0.1


def test_guess_candidates_keep_the_reference_iteration(gpu_ctx):
    """Default policy: the linear extrapolation and a network trained on the correction to it
    compete with the plain guess on the FP64 residual of the step's first Picard system, which
    stays linearised about the previous solution. The Picard iteration is then the plain one:
    the same states to the linear tolerance (1e-12 here: the two runs start their Krylov solves
    from different vectors, so their solutions differ by up to the condition number of this
    saddle-point system times that tolerance), at no more linear work."""
    from opencmp_amd.learned import GuessPolicy, MLPGuess
    from opencmp_amd.solvers import ImplicitEulerSolver
    say('guess candidates: 30 recorded steps, train (base 1), 6 compared steps')
    m = channel_model(gpu_ctx, 24, tol=1e-10)
    n = m.fes.ndof
    pol = GuessPolicy(gpu_ctx, n, max_snapshots=40)
    s = ImplicitEulerSolver(m, dt=1e-3, guess=pol)
    for _ in range(30):
        s.step()
    state = s.gfu_prev.vec.clone()
    ring = [h.clone() for h in pol.history()]
    wind = m.W.vec.clone()
    nvel = len(m.fes.comp_blocks[0])
    seg = [int(v) for v in m.fes.block_offsets()[:nvel + 1]]
    net = MLPGuess(gpu_ctx, seed=0, max_batch=16384, base=1)
    losses = net.train(pol.snapshots(), seg, steps=300, batch=16384, lr=5e-4, seed=1)
    say('  loss', losses[0], '->', losses[-1])
    assert np.isfinite(losses).all()

    def run(policy):
        mm = channel_model(gpu_ctx, 24, tol=1e-12)
        for h in reversed(ring[1:]):
            policy.push(h)
        ss = ImplicitEulerSolver(mm, dt=1e-3, gfu0=type(s.gfu_prev)(mm.fes, state.clone()), guess=policy)
        mm.W.vec.copy_(wind)
        its, first = 0, []
        for _ in range(6):
            ss.step()
            its += mm.linear_iterations
            first.append(mm.picard_log[0][0])
        return ss.gfu_prev.vec.clone(), its, first, ss.guess_log

    u_p, it_p, first_p, _ = run(GuessPolicy(gpu_ctx, n, n_learned=seg[-1]))
    u_g, it_g, first_g, log = run(GuessPolicy(gpu_ctx, n, net=net, n_learned=seg[-1], extrapolate=True))
    say(f'  plain: {it_p} iters (first Picard {first_p}); candidates: {it_g} iters (first Picard {first_g})')
    say('  choices', [(c, f'{rp:.2e}', f'{rb:.2e}') for c, rp, rb in log])
    assert len(log) == 6
    assert all(rb < rp for c, rp, rb in log if c != 'plain')
    assert sum(c != 'plain' for c, _, _ in log) >= 3
    rel = float(torch.linalg.norm(u_g - u_p) / torch.linalg.norm(u_p))
    say('  rel diff of the final states', rel)
    assert rel < 1e-5
    assert it_g <= 1.05 * it_p
    # the kept candidates carry the step's Dirichlet lift on the fixed dofs, which no solve changes
    fixed = torch.from_numpy(~m.fes.FreeDofs()).to(u_p.device)
    assert int(fixed.sum()) > 0 and torch.equal(u_g[fixed], u_p[fixed])


def test_learned_guess_saves_outer_iterations_with_schur_inner_solve(gpu_ctx):
    """The headline workload's setup (stress outlet with the no-backflow term, FGMRES + Schur inner
    PCG, mixed precision) on the channel at n=114 (450,801 dofs): 20 recorded FP64 steps, the MLP
    trained on them (base 1), then the same 4 steps from the same state with and without the learned
    guess. The guess wins the residual comparison on every step and the first Picard solve of each
    step needs fewer outer FGMRES iterations in total (the bench measures the same at n=228:
    645 against 708 outer iterations over 5 steps). The restarts make the count of one run depend on its
    rounding (355 to 411 plain over six starts 1e-13 apart, 297 to 344 learned over five of them and six
    trainings), so the totals of three starts are compared: 1,097 against 922."""
    from opencmp_amd.learned import GuessPolicy, MLPGuess
    from opencmp_amd.mesh import channel_with_holes
    from opencmp_amd.models import INS, const
    from opencmp_amd.solvers import ImplicitEulerSolver
    say('learned guess with the Schur inner solve: n=114, 20 recorded steps, 4 compared steps')
    hm = channel_with_holes(114)
    inflow = [(L.FN_POLY2, [0, 0, 6.0, 0, 0, -6.0]), const(0.0)]
    zero = [const(0.0), const(0.0)]

    def model(precision):
        return INS(hm, kv=1e-3, interp_ord=2, dirichlet={'u': {'inlet': inflow, 'wall': zero, 'cyl': zero}},
                   stress={'u': {'outlet': zero}}, linear_solver='GMRes', preconditioner='schur',
                   linear_tolerance=1e-8, restart=50, nonlinear_tolerance=(1e-6, 1e-6), nonlinear_max_iters=3,
                   precision=precision, inner_tol=1e-4 if precision == 'mixed' else 0.0, schur_iters=200,
                   schur_tol=1e-1, ctx=gpu_ctx)

    m0 = model('fp64')
    n = m0.fes.ndof
    pol = GuessPolicy(gpu_ctx, n, max_snapshots=21)
    s0 = ImplicitEulerSolver(m0, dt=1e-3, guess=pol)
    for _ in range(20):
        s0.step()
    seg = m0.fes.block_offsets()[:len(m0.fes.comp_blocks[0]) + 1]
    net = MLPGuess(gpu_ctx, seed=0, max_batch=65536, base=1)
    losses = net.train(pol.snapshots(), seg, steps=500, batch=65536, lr=5e-4, seed=1)
    say('  loss', losses[0], '->', losses[-1])
    assert losses[-1] < 0.2 * losses[0]
    state = s0.gfu_prev.vec.clone()
    ring = [h.clone() for h in pol.history()]
    wind = m0.W.vec.clone()
    del s0, m0, pol

    def run(use_net, eps):
        m = model('mixed')
        p = GuessPolicy(gpu_ctx, n, net=net if use_net else None, n_learned=seg[-1])
        for h in reversed(ring[1:]):
            p.push(h)
        s = ImplicitEulerSolver(m, dt=1e-3, gfu0=type(m.W)(m.fes, state * (1.0 + eps)), guess=p)
        m.W.vec.copy_(wind)
        first, total = [], 0
        for _ in range(4):
            r = s.step()
            assert r.converged
            first.append(m.picard_log[0][0])
            total += m.linear_iterations
        return first, total, s.guess_log, s.gfu_prev.vec.clone()

    its = {False: 0, True: 0}
    for eps in (2e-13, 1e-13, 0.0):
        fp, tp, _, up = run(False, eps)
        fl, tl, log, ul = run(True, eps)
        say(f'  first Picard solves: plain {fp} (total {tp}), learned {fl} (total {tl})')
        say('  choices', [(c, f'{rp:.2e}', f'{rl:.2e}') for c, rp, rl in log])
        assert all(c == 'learned' and rl < rp for c, rp, rl in log)
        its[False] += sum(fp)
        its[True] += sum(fl)
    assert its[True] < its[False]
    rel = float(torch.linalg.norm(ul - up) / torch.linalg.norm(up))
    say('  rel diff of the final states', rel)
    assert rel < 1e-2
