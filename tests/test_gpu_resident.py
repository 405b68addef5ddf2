"""The time loop of a problem that fits the chip (one launch for all its steps)
against the batched solver's one launch per step, bit for bit: the two share
every cell's and face's arithmetic, so no tolerance enters."""
import threading

import numpy as np
import pytest

from hyperelasticsolver_amd._lib import DomainError
from hyperelasticsolver_amd.EquationsOfState import Barton2009
from hyperelasticsolver_amd.batched import Batch
from hyperelasticsolver_amd.initial import (prim2cons, random_interfaces, random_phase_prims,
                                            random_two_phase_prims)
from hyperelasticsolver_amd.solver import Solver

pytestmark = pytest.mark.gpu

# the first and last size of every workgroup shape, teams of one and more, a
# last workgroup of a few cells, and the first size that runs step by step
SIZES = [3, 63, 65, 250, 251, 470, 1000, 59904, 59905, 123392, 123393, 250368, 250369, 377344, 377345]
STEPS, MORE = 19, 12  # past two renewals of the halo cells; then on from there


def _problem(eos, n, seed):
    rng = np.random.default_rng(seed)
    k = 6 if n > 60 else 2
    return prim2cons(eos, random_phase_prims(rng, eos, k)), random_interfaces(rng, k - 1)


def _stepwise(eos, n, flux, states, ifc, steps, t_end=None):
    with Batch([eos], [n], flux=flux) as b:
        if t_end is not None:
            b.set_t_end(t_end)
        b.set_piecewise([states], [ifc])
        b.run(steps, mode="eager")
        t, s = b.times()
        return b.get_state(), t[0], s[0]


@pytest.mark.parametrize("flux", ["rusanov", "hll", "lxf"])
@pytest.mark.parametrize("n", SIZES)
def test_resident_equals_stepwise(n, flux):
    print(f"[resident] n={n} flux={flux}", flush=True)
    eos = Barton2009() if n != 1000 else Barton2009(_beta=3.577, _gamma=2.088)
    states, ifc = _problem(eos, n, n)
    with Solver(eos, n, flux=flux) as s:
        s.set_piecewise(states, ifc)
        a = s.run(steps=STEPS, record_dt=True)
        q1 = s.get_state()
        dt = s.next_dt()
        b = s.run(steps=MORE)
        q2 = s.get_state()
    r1, t1, _ = _stepwise(eos, n, flux, states, ifc, STEPS)
    r2, t2, _ = _stepwise(eos, n, flux, states, ifc, STEPS + MORE)
    assert np.array_equal(q1, r1) and np.array_equal(q2, r2)
    assert (a["steps"], b["steps"]) == (STEPS, MORE) and (a["t"], b["t"]) == (t1, t2)
    t = 0.0
    for d in a["dt"]:
        t += d
    assert t == t1 and dt > 0.0


@pytest.mark.parametrize("flux", ["rusanov", "hll", "lxf"])
@pytest.mark.parametrize("n", [3, 15, 58, 59, 1000, 10752, 10753, 27136, 27137, 59904, 59905])
def test_resident_two_phase_equals_stepwise(n, flux):
    """Rusanov and Lax-Friedrichs to the bit; for HLL the batch sums a face's
    quadrature nodes in another order (two lanes per face, not four): 1e-13."""
    print(f"[resident two-phase] n={n} flux={flux}", flush=True)
    eos = (Barton2009(), Barton2009(_rho0=2.7, _b0=3.1))
    if n == 1000:
        eos = (Barton2009(_beta=3.577, _gamma=2.088), Barton2009(_rho0=2.7, _b0=3.1, _beta=3.577, _gamma=2.088))
    rng = np.random.default_rng(n)
    k = 6 if n > 60 else 2
    states = prim2cons(eos, random_two_phase_prims(rng, eos, k))
    ifc = random_interfaces(rng, k - 1)
    with Solver(eos, n, flux=flux) as s:
        s.set_piecewise(states, ifc)
        a = s.run(steps=STEPS, record_dt=True)
        s.run(steps=MORE)
        q = s.get_state()
    ref, t, _ = _stepwise(eos, n, flux, states, ifc, STEPS + MORE)
    assert a["steps"] == STEPS and len(a["dt"]) == STEPS
    if flux != "hll":
        assert np.array_equal(q, ref)
    else:
        assert np.all(np.abs(q - ref).max(axis=1) <= 1e-13 * np.abs(ref).max(axis=1))


@pytest.mark.parametrize("n", [200, 1000])
def test_resident_end_time(n):
    print(f"[resident t_end] n={n}", flush=True)
    eos = Barton2009()
    states, ifc = _problem(eos, n, 5)
    with Solver(eos, n, flux="rusanov") as s:
        s.set_piecewise(states, ifc)
        r = s.run(t_end=10.5 * s.next_dt())
        q = s.get_state()
        again = s.run(steps=5, t_end=r["t"])  # already there: no step
        assert again["steps"] == 0 and np.array_equal(s.get_state(), q)
    ref, t, steps = _stepwise(eos, n, "rusanov", states, ifc, 40, t_end=r["t"])
    assert np.array_equal(q, ref) and t == r["t"] and steps == r["steps"]


@pytest.mark.parametrize("n", [200, 1000, 377345])
def test_bad_state_is_reported_by_every_run(n):
    """A state outside the domain is an error of set_state and of every run
    from it, also of one that takes no step."""
    print(f"[resident bad state] n={n}", flush=True)
    eos = Barton2009()
    states, ifc = _problem(eos, n, 5)
    bad = np.array(states, order="F")
    bad[5:14, -1] *= -1.0  # det(rho A) < 0
    with Solver(eos, n, flux="rusanov") as s:
        with pytest.raises(DomainError):
            s.set_piecewise(bad, ifc)
        for call in (lambda: s.run(steps=0), lambda: s.run(steps=2), lambda: s.run(steps=0)):
            with pytest.raises(DomainError):
                call()
        s.set_piecewise(states, ifc)
        assert s.run(steps=0)["steps"] == 0 and s.run(steps=2)["steps"] == 2


def test_resident_teams_from_two_threads():
    """Two teams that each need most of the chip: one waits for the other."""
    n, eos = 200003, Barton2009()
    states, ifc = _problem(eos, n, 9)
    got = {}

    def work(k):
        with Solver(eos, n, flux="rusanov") as s:
            s.set_piecewise(states, ifc)
            for _ in range(5):
                s.run(steps=40)
            got[k] = s.get_state()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    ref, _, _ = _stepwise(eos, n, "rusanov", states, ifc, 200)
    assert np.array_equal(got[0], ref) and np.array_equal(got[1], ref)


# lengths around what one workgroup holds (one and two tiles per wave), teams,
# and a last workgroup of a few cells
LENGTHS = [3, 64, 250, 251, 498, 499, 702, 965, 1000, 5000]


@pytest.mark.parametrize("flux", ["rusanov", "hll", "lxf"])
@pytest.mark.parametrize("copies", [1, 160])  # one tile per wave; two (more than the chip at once)
def test_resident_batch_equals_stepwise(flux, copies):
    print(f"[resident batch] flux={flux} copies={copies}", flush=True)
    n = LENGTHS * copies
    general = flux == "hll" and copies == 1
    eos = [Barton2009(_b0=2.1 * (1 + 0.01 * (p % 7)), **({"_beta": 3.577, "_gamma": 2.088} if general else {}))
           for p in range(len(n))]
    data = [_problem(e, m, p % 40) for p, (e, m) in enumerate(zip(eos, n))]
    got = []
    for mode in ("eager", "graph"):
        with Batch(eos, n, flux=flux) as b:
            b.set_piecewise([d[0] for d in data], [d[1] for d in data])
            b.run(STEPS, mode=mode)
            first = b.get_state()
            t, _ = b.times()
            end = np.where(np.arange(len(n)) % 3 == 0, 1.2 * t, np.inf)  # some stop, at their own steps
            b.set_t_end(end)
            b.run(MORE, mode=mode)
            b.run(1, mode="eager")  # and on, a launch per step
            b.run(MORE, mode=mode)
            got.append((first, b.get_state(), *b.times()))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    assert got[0][3].min() < STEPS + 2 * MORE + 1 == got[0][3].max()


@pytest.mark.parametrize("mode", ["eager", "graph"])
def test_batch_goes_on_beside_a_bad_problem(mode):
    """One problem of two is outside the domain: every run says so, also one of
    no steps, and the other problem takes all its steps, in one launch or
    several."""
    print(f"[resident batch] bad problem, {mode}", flush=True)
    n, steps, eos = 20, 66000, Barton2009()
    states, ifc = _problem(eos, n, 5)
    bad = np.array(states, order="F")
    bad[5:14] *= -1.0
    with Batch([eos] * 2, [n] * 2, flux="rusanov") as b:
        with pytest.raises(DomainError):
            b.set_piecewise([states, bad], [ifc, ifc])
        for k in (0, steps, 0):
            with pytest.raises(DomainError):
                b.run(k, mode=mode)
        t, done = b.times()
        got = b.get_state()[:, :n]
    with Batch([eos], [n], flux="rusanov") as b:
        b.set_piecewise([states], [ifc])
        b.run(steps, mode="eager")
        assert done[0] == steps and t[0] == b.times()[0][0]
        assert np.array_equal(got, b.get_state())
