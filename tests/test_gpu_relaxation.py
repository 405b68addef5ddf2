"""Pressure relaxation of two-phase cells (an optional stiff source; the
reference has none, so its parity is pinned by what the mathematics fixes).

The GPU solves, per interior cell after the flux update,
    a1' - a1 = (dt / tau) (p1' - p2') / Z,   Z = sum_k rho_k c0_k^2 / a_k,
with p_k = -tr(sigma_k) / 3 of the end state, along the path on which each
phase keeps its mass, momentum and distortion shape (a rho A scaled by
(a'/a)^(1/3)) and a_k rho_k E_k changes by -p_I (a_k' - a_k), p_I the start
state's mean pressure.  It evaluates the end pressures in closed form (rho ->
rho / x, I3^(k/2) -> I3^(k/2) x^-k, W -> W x^-(beta + 4/3)).  The CPU
restatement below builds the end state itself and takes its pressures from the
oracle's cons2prim and stress (pinned against finite differences of the
energy), then finds the root with a bracketing solver; the two must agree.
On a uniform state the fluxes cancel bit for bit, so one step applies only
the source."""
import math

import numpy as np
import pytest
from scipy.optimize import brentq

from test_gpu_solver import MAT_AL, MAT_CU, _piecewise, _rand_two_phase, _two_phase_eos

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("route")]


def _pressures(ora, mats, Q):
    P = ora.cons2prim(2, mats, Q)
    out = []
    for k in range(2):
        sig = ora.stress(mats[8 * k:8 * k + 8], P[15 * k + 5], P[15 * k + 6:15 * k + 15])
        out.append(-(sig[0] + sig[4] + sig[8]) / 3.0)
    return out, P


def _end_state(Q, d, pI):
    a0, a1 = Q[0], Q[15]
    E = Q.copy()
    E[0], E[15] = a0 + d, a1 - d
    E[5] -= pI * d
    E[20] += pI * d
    E[6:15] *= np.cbrt((a0 + d) / a0)
    E[21:30] *= np.cbrt((a1 - d) / a1)
    return E


def cpu_relax(ora, mats, Q, dt, tau):
    """The implicit step from pinned pieces: end state built explicitly, its
    pressures from the oracle, the root by Brent's method."""
    (p0, p1), P = _pressures(ora, mats, Q)
    pI = 0.5 * (p0 + p1)
    Z = sum(P[15 * k + 1] * mats[8 * k + 1] ** 2 / Q[15 * k] for k in range(2))
    kc = dt / tau / Z

    def g(d):
        (q0, q1), _ = _pressures(ora, mats, _end_state(Q, d, pI))
        return d - kc * (q0 - q1)

    lo, hi = -Q[0] * (1 - 1e-12), Q[15] * (1 - 1e-12)
    d = brentq(g, lo, hi, xtol=1e-17, rtol=1e-15, maxiter=400)
    return _end_state(Q, d, pI), d


def _uniform_state(ora, rng, mats, a0=0.3):
    P = _rand_two_phase(rng, mats, 1)[:, 0]
    P[0], P[15] = a0, 1.0 - a0
    return ora.prim2cons(2, mats, P)


def _one_step(mats, q, tau, nx=64, flux="rusanov", steps=1, tau_u=None):
    from hyperelasticsolver_amd.solver import Solver
    Q0 = np.asfortranarray(np.repeat(q[:, None], nx, axis=1))
    with Solver(_two_phase_eos(mats), nx, flux=flux, cfl=0.6) as s:
        s.set_pressure_relaxation(tau)
        if tau_u is not None:
            s.set_relaxation(tau_u)
        s.set_state(Q0)
        r = s.run(steps=steps, use_graph=False, record_dt=True)
        Q = s.get_state()
    return Q, r


@pytest.mark.parametrize("flux", ["rusanov", "hll"])
def test_one_step_matches_the_cpu_restatement(ora, flux):
    """Stiff (tau << dt), moderate (tau = dt) and slow (tau = 20 dt)
    relaxation of uniform states with two materials: every interior cell
    equals the restatement's end state."""
    rng = np.random.default_rng(31)
    mats = np.concatenate([MAT_CU, MAT_AL])
    for case in range(3):
        q = _uniform_state(ora, rng, mats, a0=rng.uniform(0.2, 0.8))
        # dt of the first step (the state is uniform: the source does not change it)
        _, r0 = _one_step(mats, q, math.inf, flux=flux)
        dt = r0["dt"][0]
        for tau in (1e-15, dt, 20 * dt):
            print(f"[pressure relaxation] {flux} case {case} tau/dt {tau / dt:.1e}", flush=True)
            Q, r = _one_step(mats, q, tau, flux=flux)
            assert r["dt"][0] == dt
            ref, d = cpu_relax(ora, mats, q, dt, tau)
            assert abs(d) > 1e-6  # the source moves the volume fractions
            for i in (1, 30, 62):
                assert abs(Q[0, i] - ref[0]) <= 1e-12, (tau / dt, Q[0, i], ref[0])
                np.testing.assert_allclose(Q[:, i], ref, rtol=1e-10, atol=1e-12 * np.abs(ref).max())
            assert np.array_equal(Q[:, 0], q) and np.array_equal(Q[:, -1], q)  # frozen ends
            if tau < 1e-12:  # stiff: the step ends in pressure equilibrium
                (p0, p1), _ = _pressures(ora, mats, Q[:, 30])
                assert abs(p0 - p1) <= 1e-8 * (abs(p0) + abs(p1)), (p0, p1)


def test_equilibrium_is_a_fixed_point_and_totals_are_kept(ora):
    """A state in pressure equilibrium is left where it is; a relaxing state
    keeps the mixture's mass, momentum and total energy and a1 + a2."""
    rng = np.random.default_rng(32)
    mats = np.concatenate([MAT_CU, MAT_AL])
    print("[pressure relaxation] fixed point and totals", flush=True)
    q = _uniform_state(ora, rng, mats, a0=0.45)
    _, r0 = _one_step(mats, q, math.inf)
    dt = r0["dt"][0]
    eq, _ = cpu_relax(ora, mats, q, dt, 1e-18)  # the equilibrium reached from q
    Q, _ = _one_step(mats, eq, 1e-3 * dt)
    np.testing.assert_allclose(Q[:, 30], eq, rtol=2e-13, atol=1e-14 * np.abs(eq).max())
    # identical phases at a = 1/2: equal pressures bit for bit, nothing moves
    m2 = np.concatenate([MAT_CU, MAT_CU])
    P = _rand_two_phase(rng, m2, 1)[:, 0]
    P[15:30] = P[0:15]
    P[0] = P[15] = 0.5
    qs = ora.prim2cons(2, m2, P)
    Q, _ = _one_step(m2, qs, 1e-6)
    assert np.array_equal(Q, np.repeat(qs[:, None], Q.shape[1], axis=1))
    # totals of a relaxing cell
    Q, _ = _one_step(mats, q, 0.5 * dt)
    c = Q[:, 30]
    assert abs(c[0] - q[0]) > 1e-6
    assert c[1] == q[1] and c[16] == q[16]                      # phase masses
    assert np.array_equal(c[2:5], q[2:5]) and np.array_equal(c[17:20], q[17:20])  # momenta
    assert c[5] + c[20] == pytest.approx(q[5] + q[20], rel=1e-14, abs=1e-14)      # energy
    assert abs((c[0] + c[15]) - (q[0] + q[15])) <= 4e-16
    assert 0.0 < c[0] < 1.0 and 0.0 < c[15] < 1.0


def test_riemann_run_with_both_sources_conserves(ora):
    """A two-phase Riemann run (HLL) with velocity and pressure relaxation:
    mixture mass, momentum and energy telescope to the (equal) boundary
    fluxes, the volume fractions stay in (0, 1) with a1 + a2 kept, and with both
    sources off the step is the plain one bit for bit."""
    from hyperelasticsolver_amd.solver import Solver
    print("[pressure relaxation] Riemann run", flush=True)
    rng = np.random.default_rng(33)
    mats = np.concatenate([MAT_CU, MAT_AL])
    Ps = _rand_two_phase(rng, mats, 2)
    Ps[17:20, 0] = Ps[2:5, 0]
    Qs = ora.prim2cons(2, mats, Ps)
    # the outer state at velocity and pressure equilibrium, so that the frozen
    # end cells (which do not relax) and their neighbours stay alike
    Qs[:, 0] = cpu_relax(ora, mats, Qs[:, 0], 1.0, 1e-18)[0]
    nx = 200
    Q0 = _piecewise(nx, Qs[:, [0, 1, 0]], np.array([0.4, 0.6]))
    eos = _two_phase_eos(mats)
    out = {}
    for key, (tu, tp) in {"plain": (None, None), "off": (math.inf, math.inf),
                          "on": (2e-4, 1e-9)}.items():
        with Solver(eos, nx, flux="hll", cfl=0.6) as s:
            if tu is not None:
                s.set_relaxation(tu)
                s.set_pressure_relaxation(tp)
            s.set_state(Q0)
            s.run(steps=40, use_graph=False)
            out[key] = s.get_state()
    assert np.array_equal(out["plain"], out["off"])
    Q = out["on"]
    assert not np.array_equal(Q, out["plain"])
    assert np.all(Q[0] > 0) and np.all(Q[0] < 1) and np.all(Q[15] > 0) and np.all(Q[15] < 1)
    # the sources keep a1 + a2 of each cell to round-off
    assert np.abs(Q[0] + Q[15] - 1.0).max() <= np.abs(out["plain"][0] + out["plain"][15] - 1.0).max() + 1e-15
    for rows in ([1], [16], [2, 17], [3, 18], [4, 19], [5, 20]):
        t0 = Q0[rows].sum()
        t1 = Q[rows].sum()
        assert abs(t1 - t0) <= 1e-12 * np.abs(Q0[rows]).sum(), rows
