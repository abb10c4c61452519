"""Cases that stand for the work users of this framework have it do.

Four kinds, each through `et_amd.ccsd.CCSD` or `et_amd.solvers`:

  residual      what one ground-state iteration evaluates at given amplitudes: T1 dressing,
                Fock matrix, energy, residual (the drop-in call sequence, results on the host)
  transform     Jacobian transformations of a block of trial vectors held on the device, as
                an excited-state (right) or multiplier (left) solve passes them
  ground_state  a whole DIIS ground-state solve
  eom           a whole Davidson solve for a few roots

Sizes (n_o occupied, n_v virtual orbitals, n_J Cholesky vectors) run from one water molecule
in cc-pVDZ over (H2O)2, (H2O)4 and (H2O)8 to a basis with many virtuals per occupied orbital
close to the benchmark's own.  Inputs are random with a molecule's structure: Cholesky vectors
that decay towards the decomposition threshold and are heavier on the diagonal, a canonical
Fock matrix at t1 = 0, doubles of the MP2 form g / (energy denominators) and small singles.

Split-bf16 and FP32 results carry five to six digits; such cases return them in single
precision, which is how far a caller can use them.
"""
import numpy as np
import torch

from et_amd import ccsd, solvers

DEV = 'cuda'
GS_THRESHOLD = 1e-11
EOM_THRESHOLD = 1e-8


def _case(name, kind, n_o, n_v, n_J, precision='fp64', side='right', n_vec=1):
    c = dict(kind=kind, n_o=n_o, n_v=n_v, n_J=n_J, precision=precision, side=side, n_vec=n_vec)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one H2O / cc-pVDZ: the smallest calls, bound by launches and latency
        _case('residual_h2o', 'residual', 5, 19, 279),
        # an odd-sized molecule between one and four waters
        _case('residual_odd', 'residual', 13, 57, 601),
        # (H2O)4 / cc-pVDZ: an ordinary molecule
        _case('residual_h2o4', 'residual', 20, 76, 1270),
        # (H2O)8 / cc-pVDZ: the ground state's FP64 tail and its split-bf16 head
        _case('residual_h2o8', 'residual', 40, 152, 2541),
        _case('residual_h2o8_bf16x3', 'residual', 40, 152, 2541, 'bf16x3'),
        # many virtuals per occupied orbital: the ladder and the (ov)^3 products dominate
        _case('residual_large', 'residual', 40, 360, 1600),
        # one trial vector of one molecule: the smallest transformation
        _case('right_h2o', 'transform', 5, 19, 279, 'fp64', 'right', 1),
        # left transformations of an ordinary molecule (multipliers and left roots)
        _case('left_h2o4', 'transform', 20, 76, 1270, 'fp64', 'left', 3),
        # (H2O)8 excited states: FP64 right block, and the split-bf16 left block of the mixed solver
        _case('right_h2o8', 'transform', 40, 152, 2541, 'fp64', 'right', 7),
        _case('left_h2o8_bf16x3', 'transform', 40, 152, 2541, 'bf16x3', 'left', 12),
        # whole solves: (H2O)2 ground state, three roots of H2O-He
        _case('ground_state_h2o2', 'ground_state', 10, 38, 560),
        _case('eom_h2o_he', 'eom', 6, 23, 354, 'fp64', 'right', 3),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(['residual', 'residual', 'residual', 'transform', 'transform', 'transform',
                       'ground_state', 'eom'])
    if kind in ('ground_state', 'eom'):
        n_o = rng.randint(4, 10) if kind == 'ground_state' else rng.randint(4, 7)
        n_v = rng.randint(3 * n_o, 4 * n_o)
        n_J = rng.randint(10 * (n_o + n_v), 13 * (n_o + n_v))
        return _case(None, kind, n_o, n_v, n_J, 'fp64', rng.choice(['right', 'left']) if kind == 'eom' else 'right',
                     rng.randint(1, 4) if kind == 'eom' else 1)
    n_o = _log_uniform(rng, 4, 40)
    ratio = rng.uniform(3.0, 9.0) if kind == 'residual' else rng.uniform(3.0, 4.0)
    n_v = max(9, min(int(round(ratio * n_o)), 320 if kind == 'residual' else 152))
    n_J = rng.randint(4 * (n_o + n_v), min(12 * (n_o + n_v), max(2600, 4 * (n_o + n_v))))
    precision = rng.choice(['fp64', 'fp64', 'bf16x3', 'fp32'])
    if kind == 'residual':
        return _case(None, kind, n_o, n_v, n_J, precision)
    return _case(None, kind, n_o, n_v, n_J, precision, rng.choice(['right', 'left']),
                 rng.choice([1, 2, 3, 5, 7]) if n_o > 20 else rng.randint(1, 12))


# ---- inputs (on the device, from the seed alone) -------------------------------------------

def _inputs(case, seed):
    """L (J, p, q), h (p, q), eps (p), t1 (i, a), packed t2; L symmetric in p, q."""
    o, v, J = case['n_o'], case['n_v'], case['n_J']
    n = o + v
    g = torch.Generator(device=DEV).manual_seed(int(seed))

    def f64(*shape):
        return torch.empty(shape, dtype=torch.float64, device=DEV)

    eps = torch.cat([f64(o).uniform_(-1.5, -0.3, generator=g).sort()[0],
                     f64(v).uniform_(0.1, 3.0, generator=g).sort()[0]])
    Lt = f64(n, n, J).normal_(generator=g)                        # (q, p, J): column-major (J, p, q)
    Lt = (Lt + Lt.transpose(0, 1)).mul_(0.2 / (o * v) ** 0.5)
    ar = torch.arange(n, device=DEV)
    Lt[ar, ar] += f64(n, J).uniform_(0.0, 0.1, generator=g)
    Lt *= torch.exp(torch.arange(J, device=DEV, dtype=torch.float64) * (-8.0 / J))
    occ = Lt[:o, :, :]                                            # L(J, p, k), symmetric
    X = Lt[ar[:o], ar[:o]].sum(0)                                 # sum_k L(J, k, k)
    left = occ.permute(1, 0, 2).reshape(n, o * J)
    h = torch.diag(eps) - (2.0 * (Lt @ X) - left @ left.T)
    t1 = f64(o, v).normal_(0.0, 1e-2, generator=g)
    Lvo = Lt[:o, o:].reshape(o * v, J)                            # rows i v + a
    d = (eps[:o, None] - eps[None, o:]).reshape(-1)
    t2 = (Lvo @ Lvo.T).div_(d[:, None] + d[None, :])
    t2 = t2[torch.ones_like(t2, dtype=torch.bool).tril_()]        # packed: X (X + 1) / 2 + Y
    return dict(Lt=Lt, h=h, eps=eps, t1=t1, t2=t2)


def _amplitudes(m):
    return torch.cat([m['t1'].reshape(-1), m['t2']])


def _trials(case, seed):
    o, v = case['n_o'], case['n_v']
    N = o * v
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 7919)
    x = torch.empty((case['n_vec'], N + N * (N + 1) // 2), dtype=torch.float64, device=DEV).normal_(generator=g)
    x[:, N:] *= 1.0 / N                                            # mostly singles, as low roots are
    return x / x.norm(dim=1, keepdim=True)


def prepare(case, seed):
    m = _inputs(case, seed)
    o, v, J = case['n_o'], case['n_v'], case['n_J']
    wf = ccsd.CCSD(o, v, J)
    wf.set_cholesky(m['Lt'].cpu().numpy().T)
    wf.set_oei(m['h'].cpu().numpy())
    wf.set_orbital_energies(m['eps'].cpu().numpy())
    state = dict(case=case, wf=wf, precision=ccsd.PRECISIONS[case['precision']])
    if case['kind'] == 'ground_state':
        return state
    wf.set_amplitudes(_amplitudes(m).cpu().numpy())
    wf.construct_t1_cholesky()
    if case['kind'] in ('transform', 'eom'):
        wf.prepare_for_jacobian()
    if case['kind'] == 'transform':
        state['X'] = _trials(case, seed)
        state['R'] = torch.empty_like(state['X'])
    return state


def run(state):
    case, wf, precision = state['case'], state['wf'], state['precision']
    kind = case['kind']
    if kind == 'residual':
        wf.construct_t1_cholesky()
        F = wf.construct_fock()
        e = wf.calculate_energy()
        omega = torch.from_numpy(wf.construct_omega(precision))
        return dict(fock=F, energy=e, omega=omega if case['precision'] == 'fp64' else omega.float())
    if kind == 'transform':
        X, R = state['X'], state['R']
        wf.jacobian_transformations_at(X.data_ptr(), R.data_ptr(), case['n_vec'], case['side'], precision)
        return R if case['precision'] == 'fp64' else R.float()
    if kind == 'ground_state':
        e = solvers.DiisCCGroundState(wf, GS_THRESHOLD).run()
        return dict(energy=e, t=wf.get_amplitudes())
    e, _, X = wf.davidson(case['n_vec'], case['side'], EOM_THRESHOLD, precision=precision, vectors=True)
    return dict(energies=e, vectors=X)


# ---- work ----------------------------------------------------------------------------------

def work(case):
    """Products of the factorisation the path follows, each counted once; inputs and outputs once."""
    o, v, J = case['n_o'], case['n_v'], case['n_J']
    N, n = o * v, o + v
    op, om, vp, vm = o * (o + 1) // 2, o * (o - 1) // 2, v * (v + 1) // 2, v * (v - 1) // 2
    amps = N + N * (N + 1) // 2
    ladder = 2.0 * (op * vp ** 2 + om * vm ** 2)
    g_vvvv = 1.0 * J * v * v * (v * v + 1)
    small = 4.0 * o * o * v ** 3 + 4.0 * o ** 3 * v * v + 4.0 * o ** 4 * v * v + 2.0 * J * N * (6 * N + v)
    residual = ladder + g_vvvv + 8.0 * N ** 3 + small
    reads = 8.0 * (J * n * n + n * n + amps)
    if case['kind'] == 'residual':
        return dict(bytes=reads + 8.0 * amps, flops=residual)
    per_vector = ladder + 12.0 * N ** 3 + 2.0 * small
    if case['kind'] == 'transform':
        return dict(bytes=reads + 16.0 * amps * case['n_vec'], flops=g_vvvv + per_vector * case['n_vec'])
    if case['kind'] == 'ground_state':          # a solve takes about ten iterations
        return dict(bytes=10 * reads, flops=10 * residual)
    iterations = 12
    return dict(bytes=iterations * (reads + 16.0 * amps * case['n_vec']),
                flops=iterations * (g_vvvv + per_vector * case['n_vec']))


# ---- the same in plain torch, 64 bits ------------------------------------------------------

def _unpack(t2, N):
    full = torch.zeros((N, N), dtype=t2.dtype, device=t2.device)
    low = torch.ones((N, N), dtype=torch.bool, device=t2.device).tril()
    full = full.masked_scatter(low, t2)
    return full + full.T - torch.diag(torch.diagonal(full))


def _residual(L, h, t1, t2, o):
    """(Omega vector, Fock matrix, energy).  L (J, p, q), t1 (i, a), packed t2; T1-dressed integrals
    written out, the standard closed-shell residual equations, 1/2 on the packed diagonal."""
    J, n = L.shape[0], L.shape[1]
    v = n - o
    N = o * v
    ein = torch.einsum
    eye = torch.eye(n, dtype=L.dtype, device=L.device)
    pad = torch.nn.functional.pad
    Xm = eye - pad(t1.T, (0, v, o, 0))
    Ym = eye + pad(t1, (o, 0, 0, v))
    Lt = (Xm @ L) @ Ym.T
    oo, ov, vo, vv = Lt[:, :o, :o], Lt[:, :o, o:], Lt[:, o:, :o], Lt[:, o:, o:]
    tr = ein('Jkk->J', oo)
    F = Xm @ h @ Ym.T + 2.0 * ein('Jpq,J->pq', Lt, tr) - ein('Jpk,Jkq->pq', Lt[:, :, :o], Lt[:, :o, :])
    t = _unpack(t2, N).reshape(o, v, o, v)                         # t(i, a, j, b)
    u = 2.0 * t - t.permute(0, 3, 2, 1)
    g = (ov.reshape(J, N).T @ ov.reshape(J, N)).reshape(o, v, o, v)   # g(k, c, l, d)
    L0 = 2.0 * g - g.permute(0, 3, 2, 1)
    tau = t + ein('ia,jb->iajb', t1, t1)
    energy = (tau * L0).sum()
    # singles
    w = ein('Jkc,idkc->Jid', ov, u)
    o1 = F[o:, :o].T + ein('Jad,Jid->ia', vv, w)
    x = ein('Jlc,kalc->Jka', ov, u)
    o1 = o1 - ein('Jki,Jka->ia', oo, x) + ein('iakc,kc->ia', u, F[:o, o:])
    # doubles: E2, C2, D2 (symmetrised below)
    Fvv = F[o:, o:] - ein('kbld,ldkc->bc', u, g)
    Foo = F[:o, :o] + ein('lcjd,kdlc->kj', u, g)
    s = ein('iajc,bc->iajb', t, Fvv) - ein('iakb,kj->iajb', t, Foo)
    g_kiac = ein('Jki,Jac->iakc', oo, vv)
    g_aikc = ein('Jai,Jkc->iakc', vo, ov)
    c = g_kiac - 0.5 * ein('laid,kdlc->iakc', t, g)               # t_al,di : t(l, a, i, d)
    y = ein('kbjc,iakc->iajb', t, c)
    s = s - 0.5 * y - y.permute(2, 1, 0, 3)
    d = 2.0 * g_aikc - g_kiac + 0.5 * ein('iald,ldkc->iakc', u, L0)
    s = s + 0.5 * ein('jbkc,iakc->iajb', u, d)
    om = s + s.permute(2, 3, 0, 1)
    # A2, B2
    b = ein('Jki,Jlj->kilj', oo, oo) + ein('icjd,kcld->kilj', t, g)
    om = om + ein('Jai,Jbj->iajb', vo, vo) + ein('kalb,kilj->iajb', t, b)
    tcd = t.permute(1, 3, 0, 2).reshape(v * v, o * o)              # (c d, i j)
    flat = vv.reshape(J, v * v)
    rows = []
    for a in range(v):
        ga = (vv[:, a].T @ flat).reshape(v, v, v).permute(1, 0, 2).reshape(v, v * v)   # (b, c d)
        rows.append(ga @ tcd)
    om = om + torch.stack(rows).reshape(v, v, o, o).permute(2, 0, 3, 1)
    om = om.reshape(N, N)
    om = om - 0.5 * torch.diag(torch.diagonal(om))
    low = torch.ones((N, N), dtype=torch.bool, device=om.device).tril()
    return torch.cat([o1.reshape(-1), om.masked_select(low)]), F, energy


def exact(case, seed):
    if case['kind'] == 'eom':
        return None
    m = _inputs(case, seed)
    o, v = case['n_o'], case['n_v']
    N = o * v
    L, h, t1, t2 = m['Lt'].permute(2, 1, 0).contiguous(), m['h'], m['t1'], m['t2']
    if case['kind'] == 'residual':
        om, F, e = _residual(L, h, t1, t2, o)
        return dict(fock=F, energy=float(e), omega=om)
    if case['kind'] == 'ground_state':
        d = (m['eps'][None, o:] - m['eps'][:o, None]).reshape(-1)
        low = torch.ones((N, N), dtype=torch.bool, device=DEV).tril()
        dd = (d[:, None] + d[None, :])
        dd = (dd * (1.0 - 0.5 * torch.eye(N, dtype=dd.dtype, device=DEV))).masked_select(low)
        t1 = torch.zeros_like(t1)
        for _ in range(200):
            om, _, e = _residual(L, h, t1, t2, o)
            t1 = t1 - (om[:N] / d).reshape(o, v)
            t2 = t2 - om[N:] / dd
            if float(om.norm()) < 1e-14:
                break
        return dict(energy=float(_residual(L, h, t1, t2, o)[2]), t=torch.cat([t1.reshape(-1), t2]))
    diag = torch.arange(N, device=DEV)
    scale = torch.ones(N + t2.numel(), dtype=torch.float64, device=DEV)
    scale[N + diag * (diag + 1) // 2 + diag] = 2.0

    def omega(x):
        return _residual(L, h, x[:N].reshape(o, v), x[N:], o)[0]

    x0, out = _amplitudes(m), []
    X = _trials(case, seed)
    if case['side'] == 'right':
        for k in range(case['n_vec']):
            out.append(torch.func.jvp(omega, (x0,), (X[k] * scale,))[1])
    else:
        x0.requires_grad_(True)
        om = omega(x0)
        for k in range(case['n_vec']):
            out.append(torch.autograd.grad(om, x0, X[k], retain_graph=True)[0] * scale)
    return torch.stack(out).detach()
