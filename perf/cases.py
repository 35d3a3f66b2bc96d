"""Workloads whose speed is tracked: what a program that uses this package has it do.

Each case goes through a public entry point (``dq.mesolve``, ``dq.sesolve``,
``dq.mepropagator``, a packed DIA plan that is run again for new initial states, or
``AdjointPlan``), over the sizes that the tests, the benchmark and the documented
examples use: single small solves, ordinary batches, the largest sizes, odd dimensions,
dense and DIA operators, constant and piecewise-constant Hamiltonians, Tsit5, Dopri5,
Rouchon1 and Expm, forward solves and gradients.

``exact`` integrates the same equations in complex128 with plain torch: a Taylor series
of the flow to rounding accuracy (adaptive methods), the Kraus map itself (Rouchon1),
eigendecompositions (kets) or automatic differentiation (gradients).
"""

from __future__ import annotations

import math

import numpy as np
import torch

import dynamiqs_amd as dq
from dynamiqs_amd.adjoint import AdjointPlan
from dynamiqs_amd.integrators import dia as dia_path

KERR_T = 0.25  # solve intervals
DIA_T = 0.5
# tolerances of the solves with a few large matrix elements among many small ones: the
# absolute tolerance bounds every element, so it is set below the default 1e-6
RTOL, ATOL = 1e-6, 1e-8


def listed() -> list:
    return [
        # the first example of the documentation: one lossy oscillator, 101 saved states
        dict(name='oscillator n16', kind='oscillator', n=16, batch=1, nsave=101, dopri5=False),
        # a parameter sweep of a two-photon driven Kerr oscillator (cat-state preparation),
        # expectation values only
        dict(name='kerr n64 b128', kind='kerr', n=64, batch=128, nsave=51, dopri5=False),
        # two coupled modes small enough for one workgroup, swept over a detuning
        dict(name='two modes 9x9 b48', kind='two_mode', na=9, nb=9, batch=48, nsave=21, dopri5=False),
        # the batching tutorial: thousands of two-level Schrodinger equations in one call
        dict(name='qubits b3000', kind='kets', n=2, batch=3000, nsave=50, dopri5=False),
        # six spins with random couplings, dense Hamiltonians, a disorder average
        dict(name='kets n64 b48', kind='kets', n=64, batch=48, nsave=50, dopri5=True),
        # the serving mix at its median dimension: random dense operators
        dict(name='dense n45 k2 b64', kind='dense', n=45, jumps=2, batch=64, nsave=50, dopri5=False),
        # ... and at the upper end, where one solve is spread over the whole GPU
        dict(name='dense n233 k3 b2', kind='dense', n=233, jumps=3, batch=2, nsave=50, dopri5=False),
        # two coupled modes of 32 levels each, sparse operators, a few initial states
        dict(name='dia tsit5 32x32 b4', kind='dia_tsit5', na=32, nb=32, batch=4, nsave=6, dopri5=False),
        # the same with odd dimensions and one initial state (launches dominate)
        dict(name='dia dopri5 19x17 b1', kind='dia_tsit5', na=19, nb=17, batch=1, nsave=6, dopri5=True),
        # fixed-step positive map on the largest batch of initial states
        dict(name='dia rouchon 32x32 b16', kind='dia_rouchon', na=32, nb=32, batch=16, nsteps=40, nsave=5),
        # optimal control: gradient of a piecewise-constant drive, forward and backward solves
        dict(name='gradient n32 b64', kind='gradient', n=32, batch=64, nseg=100),
        # superoperator propagators of the documented example
        dict(name='propagator n16', kind='propagator', n=16, nint=10),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(['oscillator', 'kerr', 'two_mode', 'kets', 'dense', 'dia_tsit5', 'dia_rouchon', 'gradient',
                       'propagator'])
    dopri5 = rng.random() < 0.3
    if kind == 'oscillator':
        return dict(kind=kind, n=_log(rng, 4, 60), batch=_log(rng, 1, 12), nsave=rng.randint(11, 101), dopri5=dopri5)
    if kind == 'kerr':
        return dict(kind=kind, n=rng.randint(12, 64), batch=_log(rng, 1, 127), nsave=rng.randint(11, 51), dopri5=dopri5)
    if kind == 'two_mode':
        return dict(kind=kind, na=rng.randint(3, 10), nb=rng.randint(3, 10), batch=_log(rng, 1, 40),
                    nsave=rng.randint(5, 21), dopri5=dopri5)
    if kind == 'kets':
        n = _log(rng, 2, 200)
        return dict(kind=kind, n=n, batch=_log(rng, 1, 2900 if n < 5 else 44), nsave=rng.randint(11, 50), dopri5=dopri5)
    if kind == 'dense':
        n = _log(rng, 8, 220)
        return dict(kind=kind, n=n, jumps=rng.randint(1, 3), batch=_log(rng, 1, 60 if n < 96 else 2),
                    nsave=rng.randint(11, 50), dopri5=dopri5)
    if kind == 'dia_tsit5':
        return dict(kind=kind, na=rng.randint(12, 31), nb=rng.randint(12, 32), batch=rng.randint(1, 4),
                    nsave=rng.randint(3, 6), dopri5=dopri5)
    if kind == 'dia_rouchon':
        return dict(kind=kind, na=rng.randint(12, 31), nb=rng.randint(12, 32), batch=rng.randint(1, 15),
                    nsteps=4 * rng.randint(5, 10), nsave=5)
    if kind == 'gradient':
        return dict(kind=kind, n=rng.randint(8, 31), batch=rng.randint(8, 60), nseg=10 * rng.randint(2, 9))
    return dict(kind=kind, n=rng.randint(6, 15), nint=rng.randint(4, 10))


# ------------------------------------------------------------------------- inputs
def _two_mode(na: int, nb: int):
    a = dq.tensor(dq.destroy(na), dq.eye(nb))
    b = dq.tensor(dq.eye(na), dq.destroy(nb))
    ad, bd = a.dag(), b.dag()
    H = 5.0 * (ad @ a) + 6.0 * (bd @ b) + 0.1 * (ad @ b + a @ bd) - 0.01 * (ad @ a @ bd @ b)
    return H, [math.sqrt(0.02) * a, math.sqrt(0.05) * b], a, b


def _coherent(n: int, alpha) -> np.ndarray:
    """Normalised truncated coherent state(s) (..., n) from the number-state amplitudes."""
    alpha = np.asarray(alpha, dtype=np.complex128)
    k = np.arange(n)
    logf = np.concatenate([[0.0], np.cumsum(np.log(np.arange(1, n)))])
    c = np.power(alpha[..., None], k) * np.exp(-0.5 * logf)
    return c / np.linalg.norm(c, axis=-1, keepdims=True)


def _build(case, seed: int) -> dict:
    """Arguments of the call, as host objects, from the seed alone."""
    rng = np.random.default_rng(seed)
    kind = case['kind']
    if kind == 'oscillator':
        n, B = case['n'], case['batch']
        a = dq.destroy(n)
        w = rng.uniform(0.8, 1.2, size=B)
        eps = rng.uniform(0.1, 0.3)
        alpha = min(1.0, 0.2 * math.sqrt(n)) * np.exp(1j * rng.uniform(0, 2 * np.pi))
        num = a.dag() @ a
        H = (w[0] if B == 1 else w[:, None, None]) * num + eps * (a + a.dag())
        return dict(H=H, Ls=[math.sqrt(0.1) * a], y0=_coherent(n, alpha)[:, None],
                    tsave=np.linspace(0.0, 2 * np.pi, case['nsave']), exp_ops=[num], save_states=True)
    if kind == 'kerr':
        n, B = case['n'], case['batch']
        a = dq.destroy(n)
        ad = a.dag()
        a2, ad2 = a @ a, ad @ ad
        eps = rng.uniform(0.5, 4.0, size=B)
        H = -1.0 * (ad2 @ a2) + eps[:, None, None] * (a2 + ad2)
        return dict(H=H, Ls=[0.1 * a, 1.0 * a2], y0=_coherent(n, 0.1 * rng.normal())[:, None],
                    tsave=np.linspace(0.0, KERR_T, case['nsave']), exp_ops=[ad @ a, a2], save_states=False)
    if kind == 'two_mode':
        na, nb, B = case['na'], case['nb'], case['batch']
        H, Ls, a, b = _two_mode(na, nb)
        det = rng.uniform(-0.5, 0.5, size=B)
        H = H + det[:, None, None] * (b.dag() @ b)
        psi = np.kron(_coherent(na, rng.uniform(0.3, 0.8)), _coherent(nb, rng.uniform(0.3, 0.8)))
        return dict(H=H, Ls=Ls, y0=psi[:, None], tsave=np.linspace(0.0, 1.0, case['nsave']),
                    exp_ops=[a.dag() @ a, b], save_states=True)
    if kind == 'kets':
        n, B = case['n'], case['batch']
        A = rng.normal(size=(B, n, n)) + 1j * rng.normal(size=(B, n, n))
        H = 0.5 * (A + np.swapaxes(A.conj(), -1, -2)) / math.sqrt(n)
        psi = rng.normal(size=n) + 1j * rng.normal(size=n)
        E = rng.normal(size=(n, n))
        return dict(H=H, Ls=None, y0=(psi / np.linalg.norm(psi))[:, None],
                    tsave=np.linspace(0.0, 1.0 if n < 5 else 5.0, case['nsave']), exp_ops=[0.5 * (E + E.T)],
                    save_states=True)
    if kind == 'dense':
        n, B, K = case['n'], case['batch'], case['jumps']
        A = rng.normal(size=(B, n, n)) + 1j * rng.normal(size=(B, n, n))
        H = 0.5 * (A + np.swapaxes(A.conj(), -1, -2)) / (2.0 * math.sqrt(n))  # spectral norm about 1
        Ls = [math.sqrt(rng.uniform(0.01, 0.5) / (2 * n)) * (rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n)))
              for _ in range(K)]
        psi = rng.normal(size=n) + 1j * rng.normal(size=n)
        return dict(H=H, Ls=Ls, y0=(psi / np.linalg.norm(psi))[:, None], tsave=np.linspace(0.0, 8.0, case['nsave']),
                    exp_ops=[np.diag(np.arange(n) / n)], save_states=n > 100)
    if kind in ('dia_tsit5', 'dia_rouchon'):
        na, nb, B = case['na'], case['nb'], case['batch']
        H, Ls, a, b = _two_mode(na, nb)
        alpha = rng.uniform(0.5, 2.0, size=B)
        psi = np.stack([np.kron(_coherent(na, x), _coherent(nb, 0.3)) for x in alpha])
        T = DIA_T if kind == 'dia_tsit5' else 1e-3 * case['nsteps']
        return dict(H=H, Ls=Ls, y0=psi, tsave=np.linspace(0.0, T, case['nsave']), exp_ops=[a.dag() @ a])
    if kind == 'gradient':
        n, B, nseg = case['n'], case['batch'], case['nseg']
        a = np.diag(np.sqrt(np.arange(1, n, dtype=np.float64)), k=1).astype(np.complex128)
        rho0 = np.zeros((n, n), dtype=np.complex128)
        rho0[0, 0] = 1.0
        return dict(H=a.conj().T @ a, X=a + a.conj().T, Ls=[math.sqrt(0.05) * a], y0=rho0,
                    times=0.1 * np.arange(nseg + 1), u=rng.normal(0.0, 0.5, size=(B, 1, nseg)))
    n = case['n']
    a = dq.destroy(n)
    return dict(H=rng.uniform(0.8, 1.2) * (a.dag() @ a) + rng.uniform(0.1, 0.3) * (a + a.dag()), Ls=[1.0 * a],
                tsave=np.linspace(0.0, 1.0, case['nint'] + 1))


def prepare(case, seed) -> dict:
    d = _build(case, seed)
    kind = case['kind']
    state = dict(kind=kind, args=d)
    if kind in ('oscillator', 'kerr', 'two_mode', 'kets', 'dense'):
        tol = dq.method.Dopri5 if case['dopri5'] else dq.method.Tsit5
        # the serving mix asks for 1e-5, the tutorials' Schrodinger equations take the defaults
        state['method'] = (tol(rtol=1e-5) if kind == 'dense' else tol() if kind == 'kets'
                           else tol(rtol=RTOL, atol=ATOL))
        state['options'] = dq.Options(save_states=d['save_states'])
    elif kind in ('dia_tsit5', 'dia_rouchon'):
        H, Ls = d['H'].to_numpy().astype(np.complex128), [L.to_numpy().astype(np.complex128) for L in d['Ls']]
        rho = np.einsum('bi,bj->bij', d['y0'], d['y0'].conj())
        Es = [E.to_numpy() for E in d['exp_ops']]
        if kind == 'dia_tsit5':
            state['plan'] = dia_path.tsit5_plan(H, Ls, rho, d['tsave'], exp_ops=Es, rtol=RTOL, atol=ATOL,
                                                tableau='dopri5' if case['dopri5'] else 'tsit5')
        else:
            state['plan'] = dia_path.build_plan(H, Ls, rho, d['tsave'], 1e-3, exp_ops=Es)
    elif kind == 'gradient':
        state['plan'] = AdjointPlan(d['H'], [d['X']], d['times'], d['Ls'], d['y0'], d['H'], case['batch'],
                                    checkpoint_every=10)
    return state


def run(state):
    kind, d = state['kind'], state['args']
    if kind in ('oscillator', 'kerr', 'two_mode', 'dense'):
        r = dq.mesolve(d['H'], d['Ls'], d['y0'], d['tsave'], exp_ops=d['exp_ops'], method=state['method'],
                       options=state['options'])
        return [r.states.to_numpy(), r.expects]
    if kind == 'kets':
        r = dq.sesolve(d['H'], d['y0'], d['tsave'], exp_ops=d['exp_ops'], method=state['method'],
                       options=state['options'])
        return [r.states.to_numpy(), r.expects]
    if kind in ('dia_tsit5', 'dia_rouchon'):
        plan = state['plan']
        plan.reset()
        plan.run()
        return [plan.states, plan.expects]  # complex64 as float32 pairs, on the GPU
    if kind == 'gradient':
        r = state['plan'].run(d['u'])
        return [r.J, r.grad_u, r.lambda0]
    return [dq.mepropagator(d['H'], d['Ls'], d['tsave']).propagators.to_numpy()]


# ------------------------------------------------------------------------ accounting
def work(case) -> dict:
    """Inputs and outputs once; for the adaptive methods the vector fields of about the
    steps that the default tolerances take, with the products that the operators' nonzero
    diagonals need."""
    kind = case['kind']
    if kind in ('kets', 'dense', 'oscillator', 'kerr'):
        n, B, S = case['n'], case['batch'], case['nsave']
    if kind == 'kets':
        rhs = 6 * (12 if n < 5 else 40)
        return dict(bytes=8.0 * B * (n * n + S * n + S), flops=8.0 * B * rhs * n * n)
    if kind == 'dense':
        K = case['jumps']
        out = (S if n > 100 else 1) * n * n
        return dict(bytes=8.0 * (B * (n * n + out) + K * n * n), flops=8.0 * B * 6 * 30 * (1 + 2 * K) * n**3)
    if kind == 'oscillator':  # H and L on 4 diagonals: about 7 products per element
        return dict(bytes=8.0 * B * (S * n * n + 3 * n), flops=8.0 * B * 6 * 60 * 7 * n * n)
    if kind == 'kerr':
        steps = max(20.0, 0.11 * KERR_T * n * n)
        return dict(bytes=8.0 * B * (n * n + 2 * S + 3 * n), flops=8.0 * B * 6 * steps * 8 * n * n)
    if kind == 'two_mode':
        n, B, S = case['na'] * case['nb'], case['batch'], case['nsave']
        return dict(bytes=8.0 * B * (S * n * n + 3 * n), flops=8.0 * B * 6 * 40 * 8 * n * n)
    if kind == 'dia_tsit5':
        n, B, S = case['na'] * case['nb'], case['batch'], case['nsave']
        rhs = 6 * 0.12 * DIA_T * (5 * case['na'] + 6 * case['nb'])
        # every vector field reads a state and writes one
        return dict(bytes=8.0 * B * n * n * (2 * rhs + S), flops=8.0 * B * rhs * 8 * n * n)
    if kind == 'dia_rouchon':
        n, B = case['na'] * case['nb'], case['batch']
        return dict(bytes=8.0 * B * n * n * (2 * case['nsteps'] + case['nsave']),
                    flops=8.0 * B * case['nsteps'] * 17 * n * n)
    if kind == 'gradient':
        n, B, nseg = case['n'], case['batch'], case['nseg']
        return dict(bytes=8.0 * B * (2 * nseg + n * n), flops=8.0 * B * 3 * 6 * nseg * 7 * n * n)
    N, k = case['n'] ** 2, case['nint']
    return dict(bytes=8.0 * N * N * (1 + k), flops=8.0 * N**3 * (10 + k - 1))


def tolerance(case) -> dict:
    """About four times the largest difference measured between two evaluations at the
    same precision: another kernel form (sums in another order), and operators perturbed
    by one FP32 rounding, which also moves the adaptive steps."""
    rel, largest = {
        'oscillator': (1e-6, 4e-5),
        'kerr': (2e-6, 4e-4),
        'two_mode': (2e-6, 2e-4),
        'kets': (2e-6, 4e-5),
        'dense': (8e-6, 4e-4),
        'dia_tsit5': (8e-6, 5e-3),
        'dia_rouchon': (1.2e-7, 2e-5),
        'gradient': (2e-6, 2e-4),
        'propagator': (3e-6, 5e-5),  # against the matrix exponential in complex128
    }[case['kind']]
    return dict(rel=rel, max=largest)


# --------------------------------------------------------------------- 64-bit results
def _dev(x):
    return torch.as_tensor(np.ascontiguousarray(np.asarray(x, dtype=np.complex128)),
                           device='cuda' if torch.cuda.is_available() else 'cpu')


def _np(q):
    return q.to_numpy() if hasattr(q, 'to_numpy') else np.asarray(q)


def _flow(f, y, h: float, bound: float):
    """exp(h f) y of a linear field by Taylor series on substeps of length <= 4 / bound."""
    m = max(1, int(math.ceil(h * bound / 4.0)))
    dt = h / m
    for _ in range(m):
        term = y
        for k in range(1, 41):
            term = f(term) * (dt / k)
            y = y + term
    return y


def _lindblad(G, Ls):
    def f(r):
        t = G @ r
        out = t + t.mH
        for L in Ls:
            out = out + L @ r @ L.mH
        return out

    return f


def _master(H, Ls, rho, tsave, Es):
    """States (B, nsave, n, n) and Tr(E rho) (B, nE, nsave) of dense complex128 inputs."""
    H, rho, Es = _dev(H), _dev(rho), _dev(Es)
    Ls = [_dev(L) for L in Ls]
    H = H if H.ndim == 3 else H[None]
    B = max(len(H), len(rho))
    rho = rho.expand(B, -1, -1).contiguous()
    G = -1j * H - 0.5 * sum((L.mH @ L for L in Ls), torch.zeros_like(H[0]))
    bound = 2 * float(torch.linalg.matrix_norm(G, 1).max()) ** 0.5 * float(torch.linalg.matrix_norm(G, float('inf')).max()) ** 0.5
    bound += sum(float(torch.linalg.matrix_norm(L, 1) * torch.linalg.matrix_norm(L, float('inf'))) for L in Ls)
    f = _lindblad(G, Ls)
    states = [rho]
    for h in np.diff(tsave):
        rho = _flow(f, rho, float(h), bound)
        states.append(rho)
    states = torch.stack(states, dim=1)
    ex = torch.einsum('eij,btji->bet', Es, states)
    return states, ex


def _flat(x):
    """complex64-as-float32-pairs layout of a plan's buffers, in 64 bits."""
    return torch.view_as_real(x.contiguous()).reshape(-1).cpu().numpy()


def exact(case, seed):
    d = _build(case, seed)
    kind = case['kind']
    if kind in ('oscillator', 'kerr', 'two_mode', 'dense'):
        psi = np.asarray(d['y0'])
        st, ex = _master(_np(d['H']), [_np(L) for L in d['Ls']], (psi @ psi.conj().T)[None], d['tsave'],
                         np.stack([_np(E) for E in d['exp_ops']]))
        if not d['save_states']:
            st = st[:, -1:]
        if np.ndim(_np(d['H'])) == 2:
            st, ex = st[0], ex[0]
        return [st.cpu().numpy(), ex.cpu().numpy()]
    if kind == 'kets':
        w, V = torch.linalg.eigh(_dev(d['H']).cpu())
        c = V.mH @ _dev(d['y0']).cpu()
        t = torch.as_tensor(d['tsave'])
        ph = torch.exp(-1j * w[:, None, :] * t[None, :, None])
        st = torch.einsum('bij,btj->bti', V, ph * c[:, None, :, 0])
        E = _dev(d['exp_ops'][0]).cpu()
        ex = torch.einsum('bti,ij,btj->bt', st.conj(), E, st)[:, None]
        return [st[..., None].numpy(), ex.numpy()]
    if kind == 'dia_tsit5':
        rho = np.einsum('bi,bj->bij', d['y0'], d['y0'].conj())
        st, ex = _master(_np(d['H']), [_np(L) for L in d['Ls']], rho, d['tsave'],
                         np.stack([_np(E) for E in d['exp_ops']]))
        return [_flat(st), _flat(ex)]
    if kind == 'dia_rouchon':
        dt = 1e-3
        H, Ls = _dev(_np(d['H'])), [_dev(_np(L)) for L in d['Ls']]
        E = _dev(_np(d['exp_ops'][0]))
        eye = torch.eye(len(H), dtype=H.dtype, device=H.device)
        LdL = sum(L.mH @ L for L in Ls)
        Ms = [eye - dt * (1j * H + 0.5 * LdL)] + [math.sqrt(dt) * L for L in Ls]
        T = torch.linalg.cholesky(sum(M.mH @ M for M in Ms))
        Tdi = torch.linalg.solve_triangular(T, eye, upper=False).mH
        Ms = [M @ Tdi for M in Ms]
        rho = _dev(np.einsum('bi,bj->bij', d['y0'], d['y0'].conj()))
        every = case['nsteps'] // (case['nsave'] - 1)
        states = [rho]
        for m in range(1, case['nsteps'] + 1):
            rho = sum(M @ rho @ M.mH for M in Ms)
            if m % every == 0:
                states.append(rho)
        st = torch.stack(states, dim=1)
        return [_flat(st), _flat(torch.einsum('ij,btji->bt', E, st))]
    if kind == 'gradient':
        H, X, L, O = _dev(d['H']), _dev(d['X']), _dev(d['Ls'][0]), _dev(d['H'])
        u = torch.as_tensor(d['u'][:, 0], device=H.device).requires_grad_()
        rho0 = _dev(d['y0'])[None].repeat(case['batch'], 1, 1).requires_grad_()
        rho, LdL = rho0, L.mH @ L
        for k in range(case['nseg']):
            Gk = -1j * (H + u[:, k, None, None] * X) - 0.5 * LdL

            def f(r, Gk=Gk):
                return Gk @ r + r @ Gk.mH + L @ r @ L.mH

            rho = _flow(f, rho, 0.1, 2.0 * case['n'] + 20.0)
        J = torch.einsum('ij,bji->b', O, rho).real
        J.sum().backward()
        # dJ = Tr(lambda drho0), so lambda is the Hermitian part of the gradient
        lam = 0.5 * (rho0.grad + rho0.grad.mH)
        return [J.detach().cpu().numpy(), u.grad[:, None].cpu().numpy(), lam.cpu().numpy()]
    H, Ls = _dev(_np(d['H'])), [_dev(_np(L)) for L in d['Ls']]
    n = len(H)
    eye = torch.eye(n, dtype=H.dtype, device=H.device)
    G = -1j * H - 0.5 * sum(L.mH @ L for L in Ls)
    S = torch.kron(eye, G) + torch.kron(G.conj(), eye) + sum(torch.kron(L.conj(), L) for L in Ls)
    dt = float(d['tsave'][1] - d['tsave'][0])
    P = torch.matrix_exp(S.cpu() * dt)
    U = [torch.eye(n * n, dtype=H.dtype)]
    for _ in range(case['nint']):
        U.append(P @ U[-1])
    return [torch.stack(U).numpy()]
