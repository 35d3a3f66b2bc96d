"""GPU parity of the few-diagonal Tsit5 / Dopri5 kernel (``dqh_mesolve_tsit5_diag``)
against the complex128 oracle replaying the GPU's own accepted steps, at the edges of its
size classes (64, 192 and 576 threads with one element, then two and three elements per
thread; with tables up to n = 90 in registers and above in memory), with no, one and many
shifts, far offsets, and with PWC and modulated terms."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _banded(rng, n, offs, scale=1.0):
    x = np.zeros((n, n), dtype=np.complex128)
    for o in offs:
        m = n - abs(o)
        if m > 0:
            x += scale * np.diag(rng.normal(size=m) + 1j * rng.normal(size=m), k=o)
    return x


def _drive(t):
    return 0.7 * np.cos(5.0 * t)


def _insts(n, offH, offL, B, pwc=False, mod=False):
    from dynamiqs_amd.integrators.dense import Instance

    rng = np.random.default_rng(n + len(offH))
    Ls = [_banded(rng, n, o, 0.3) for o in offL]
    out = []
    for b in range(B):
        H = _banded(rng, n, offH)
        psi = rng.normal(size=(n, 1)) + 1j * rng.normal(size=(n, 1))
        psi /= np.linalg.norm(psi)
        X = _banded(rng, n, [1, 0])
        terms = [(np.array([0.1, 0.5, 0.8]), rng.normal(size=2) + 0j, X + X.conj().T)] if pwc else []
        mods = [(_drive, X + X.conj().T, ('drive',))] if mod else []
        out.append(Instance(H=H + H.conj().T, Ls=Ls, rho0=psi @ psi.conj().T, pwc=terms, mod=mods, key_H=(b,), key_L=(), key_rho=(b,)))
    return out


def _replay(inst, tsave, ends, method):
    from oracle import lindblad, tsit5

    def f(t, y, tseg):
        H = inst.H
        for times, vals, op in inst.pwc:
            if times[0] <= tseg < times[-1]:
                H = H + vals[np.searchsorted(times, tseg, side='right') - 1] * op
        for g, op, _ in inst.mod:
            H = H + g(t) * op
        return lindblad.rhs_hermitian(H, inst.Ls, y)

    kw = dict(tab=tsit5.tableau('dopri5')) if method == 'dopri5' else {}
    saved, _ = tsit5.integrate_steps(f, inst.rho0, tsave, ends, **kw)
    return np.stack(saved)


CASES = [
    (1, [0], [[0]], 'tsit5'), (2, [-1, 0, 1], [[1]], 'dopri5'), (10, [-1, 0, 1], [[1], [0]], 'tsit5'),
    (11, [0], [[-1, 1]], 'tsit5'), (16, [-1, 0, 1], [[1]], 'tsit5'), (19, [0], [], 'tsit5'), (20, [-2, 2], [[2], [1]], 'dopri5'),
    (33, [-1, 0, 1], [[1], [-1], [0]], 'tsit5'), (34, [-5, -1, 0, 1, 5], [[1], [5]], 'tsit5'),
    (47, [0, 1], [[1]], 'tsit5'), (48, [-1, 1], [[2]], 'dopri5'), (64, [-2, 0, 2], [[1], [2]], 'tsit5'),
    (64, [-8, -1, 0, 1, 8], [[1], [8], [0]], 'tsit5'),
    # the table form: far offsets, many pairs, sizes above 64
    (64, [-62, 62], [[62], [-60]], 'tsit5'), (20, [0, 1], [[0, 1, 2], [1]], 'dopri5'), (63, [-1, 1], [[-1, 0, 1], [5]], 'tsit5'),
    (65, [-8, -1, 0, 1, 8], [[1], [8]], 'tsit5'), (90, [-9, 9], [[9], [1], [0]], 'dopri5'),
    (91, [-10, 10], [[10], [0, 1]], 'tsit5'), (127, [-1, 0, 1], [[1], [126]], 'tsit5'),
    # the last of one and the first of the next number of elements per thread
    (74, [-1, 1], [[1]], 'tsit5'), (75, [-1, 1], [[1]], 'dopri5'), (83, [-9, 9], [[9], [0, 1]], 'tsit5'),
    (84, [-1, 1], [[1], [83]], 'tsit5'), (100, [-10, 10], [[10], [1]], 'dopri5'), (101, [-1, 0, 1], [[1]], 'tsit5'),
    (110, [-1, 1], [[1]], 'tsit5'), (111, [-1, 1], [[2]], 'dopri5'),
]


@pytest.mark.parametrize('n,offH,offL,method', CASES)
def test_matches_fp64_replay(n, offH, offL, method):
    from dynamiqs_amd.integrators import dense

    tsave = np.linspace(0.0, 1.0, 6)
    for pwc, mod in ((False, False), (True, False), (True, True)):
        insts = _insts(n, offH, offL, 3, pwc, mod)
        E = np.diag(np.arange(n)) + 0j
        plan = dense.build_plan('tsit5', insts, tsave, exp_ops=[E], rtol=1e-6, atol=1e-8, step_log_cap=4000,
                                tableau=method, dia_ops=True)
        assert plan.stencil is not None
        plan.run()
        out = plan.results()
        assert np.all(out['status'] == 0)
        for b, inst in enumerate(insts):
            ref = _replay(inst, tsave, out['step_ends'][b], method)
            # FP32 stages: about nsteps^(1/2) roundings of 6e-8 (the dense kernels' replay bar)
            assert np.linalg.norm(out['states'][b] - ref, axis=(-2, -1)).max() <= 2e-6, (n, pwc, mod, b)
            assert np.abs(out['expects'][b, 0] - np.einsum('ij,tji->t', E, out['states'][b])).max() <= 1e-5 * n
            assert np.array_equal(out['states'][b], np.swapaxes(out['states'][b].conj(), -1, -2))
            assert np.array_equal(out['final_state'][b], out['states'][b, -1])
        if not mod:
            # the step sequence of the dense kernels up to rounding. (With modulated terms the
            # stages are evaluated at the full state, and their FP32 rounding, 6e-8 |f| each,
            # is of the size of atol in the error estimate, so the sequences differ.)
            dplan = dense.build_plan('tsit5', insts, tsave, rtol=1e-6, atol=1e-8, tableau=method)
            dplan.run()
            assert np.all(np.abs(dplan.results()['nsteps'] - out['nsteps']) <= 2)
        # bit-identical alone
        solo = dense.build_plan('tsit5', insts[1:2], tsave, rtol=1e-6, atol=1e-8, tableau=method, dia_ops=True)
        solo.run()
        assert np.array_equal(solo.results()['states'][0], out['states'][1])


def test_mesolve_takes_dia_operators_there_and_stops_as_before():
    import dynamiqs_amd as dq
    from dynamiqs_amd.integrators import dense

    a = dq.destroy(12)
    seen = []
    run = dense.DensePlan.run
    dense.DensePlan.run = lambda self, *s: (seen.append(self.stencil is not None), run(self, *s))[1]
    try:
        kw = dict(exp_ops=[a.dag() @ a], options=dq.Options(save_states=False))
        r = dq.mesolve(a.dag() @ a + 0.2 * (a + a.dag()), [a], dq.fock(12, 3), np.linspace(0, 1, 5), **kw)
        rd = dq.mesolve((a.dag() @ a + 0.2 * (a + a.dag())).asdense(), [a.asdense()], dq.fock(12, 3), np.linspace(0, 1, 5), **kw)
        with pytest.raises(RuntimeError, match='maximum number of method steps'):
            dq.mesolve(a.dag() @ a, [a], dq.fock(12, 3), np.linspace(0, 9, 3), method=dq.method.Tsit5(max_steps=3))
        H = a.dag() @ a
        nan = H * np.nan
        with pytest.raises(RuntimeError, match='non-finite'):
            dq.mesolve(nan, [a], dq.fock(12, 3), np.linspace(0, 1, 3))
    finally:
        dense.DensePlan.run = run
    assert seen == [True, False, True, True]
    assert np.abs(r.expects - rd.expects).max() <= 1e-6 and r.states.shape == rd.states.shape
    assert np.linalg.norm(r.states.to_numpy() - rd.states.to_numpy()) <= 1e-6


@pytest.mark.parametrize('n', [3, 40, 64, 70, 100])
def test_saves_after_an_early_stop_are_the_state(n):
    """A first attempt whose stages overflow FP32 (a coupling of 1e28 that the initial state
    does not touch) is rejected and max_steps = 1 ends the solve there: the saves not reached
    are the initial state, as final_state is, in every form of the kernel."""
    from dynamiqs_amd import _native
    from dynamiqs_amd.integrators import dense

    H = np.zeros((n, n), dtype=np.complex128)
    H[0, 1] = H[1, 0] = 1.0
    H[1, 2] = H[2, 1] = 1e28
    rho0 = np.zeros((n, n), dtype=np.complex128)
    rho0[0, 0] = 1.0
    E = np.diag(np.arange(1.0, n + 1)) + 0j
    plan = dense.build_plan('tsit5', [dense.Instance(H=H, Ls=[np.diag(np.ones(n - 1), 1) + 0j], rho0=rho0)],
                            np.linspace(0.0, 1.0, 4), exp_ops=[E], max_steps=1, dia_ops=True)
    assert plan.stencil is not None
    plan.run()
    out = plan.results()
    assert out['status'][0] == _native.STATUS_MAX_STEPS and out['nrejected'][0] == 1
    assert np.array_equal(out['final_state'][0], rho0.astype(np.complex64))
    assert np.array_equal(out['states'][0], np.broadcast_to(rho0.astype(np.complex64), (4, n, n)))
    assert np.array_equal(out['expects'][0, 0], np.ones(4))
