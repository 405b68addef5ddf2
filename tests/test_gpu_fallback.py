"""What follows when the workgroups of a one-launch time loop do not meet: the
launch ends at its own bounded wait (a wait of no time, set from the host) and
the run goes on with a launch per step.  Against runs that take a launch per
step from the start, bit for bit (the same arithmetic)."""
import numpy as np
import pytest

from hyperelasticsolver_amd.EquationsOfState import Barton2009
from hyperelasticsolver_amd.adjoint import Adjoint, BatchAdjoint, phase_prims_to_adjoint
from hyperelasticsolver_amd.batched import Batch
from hyperelasticsolver_amd.initial import (prim2cons, random_interfaces, random_phase_prims,
                                            random_two_phase_prims)
from hyperelasticsolver_amd.solver import Solver

pytestmark = pytest.mark.gpu

EOS = Barton2009()
EOS2 = (Barton2009(), Barton2009(_rho0=2.7, _b0=3.1))
WAIT = 4_000_000


# teams of several workgroups of every shape (threads, tiles per wave)
@pytest.mark.parametrize("nph,n,flux", [(1, 1000, "rusanov"), (1, 1000, "hll"), (1, 60000, "lxf"),
                                        (1, 130000, "hll"), (1, 300000, "rusanov"),
                                        (2, 1000, "rusanov"), (2, 1000, "hll"), (2, 20000, "hll"),
                                        (2, 30000, "lxf")])
def test_solver(nph, n, flux):
    print(f"[fallback] solver nph={nph} n={n} {flux}", flush=True)
    eos = EOS if nph == 1 else EOS2
    rng = np.random.default_rng(n)
    states = prim2cons(eos, (random_phase_prims if nph == 1 else random_two_phase_prims)(rng, eos, 5))
    ifc = random_interfaces(rng, 4)

    def run(waits):
        """Four stretches of steps, the team's wait set before each."""
        out = []
        with Solver(eos, n, flux=flux) as s:
            if nph == 2:
                s.set_relaxation(1e-3)
                s.set_pressure_relaxation(1e-3)
            s.set_piecewise(states, ifc)
            for steps, wait in zip((13, 70, 9, 20), waits):
                before = s.team(wait)
                r = s.run(steps=steps, record_dt=steps < 60)
                out.append((s.get_state(), r["t"], r["steps"], s.next_dt(), s.get_speeds(), r.get("dt")))
                team = s.team()
                assert team == (0 if wait <= 0 else before) and (before > 1) == (wait >= 0)
            # no step to take, and a team that gives up all the same
            s.team(0)
            r = s.run(steps=5, t_end=out[-1][1])
            assert r["steps"] == 0 and r["t"] == out[-1][1] and s.team() == 0
            assert np.array_equal(s.get_state(), out[-1][0]) and s.next_dt() == out[-1][3]
            s.run(steps=3)
            out.append((s.get_state(),))
        return out

    ref = run((-1, -1, -1, -1))
    for waits in ((0, -1, WAIT, 0), (WAIT, 0, WAIT, -1), (WAIT, -1, 0, WAIT)):
        for a, b in zip(run(waits), ref):
            for x, y in zip(a, b):
                assert np.array_equal(x, y) if x is not None else y is None


@pytest.mark.parametrize("flux", ["rusanov", "hll"])
@pytest.mark.parametrize("copies", [1, 100])  # one tile per wave; two, more than the chip at once
def test_batch(flux, copies):
    print(f"[fallback] batch {flux} x {copies}", flush=True)
    cells = [3, 250, 700, 1000, 5000] * copies
    rng = np.random.default_rng(copies)
    states = [prim2cons(EOS, random_phase_prims(rng, EOS, 2)) for _ in cells]

    def run(waits):
        out = []
        with Batch([EOS] * len(cells), cells, flux=flux) as b:
            b.set_piecewise(states, [[0.5]] * len(cells))
            for steps, wait in zip((13, 30, 20), waits):
                before = b.team(wait)
                b.run(steps)
                assert b.team() == (0 if wait <= 0 else before) and (before > 0) == (wait >= 0)
                t, k = b.times()
                out.append((b.get_state(), t, k))
                b.set_t_end(np.where(np.arange(len(cells)) % 3 == 0, 1.2 * t, np.inf))
        return out

    ref = run((-1, -1, -1))
    for waits in ((0, -1, WAIT), (WAIT, 0, WAIT)):
        for a, b in zip(run(waits), ref):
            assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("n", [1000, 50000])
def test_adjoint(n, graph):
    print(f"[fallback] adjoint n={n} graph={graph}", flush=True)
    rng = np.random.default_rng(n)
    prims = phase_prims_to_adjoint(random_phase_prims(rng, EOS, 3))

    def run(wait):
        with Adjoint(EOS, n, 60, every=20) as a:
            a.set_launch(graph)
            assert (a.team(wait) > 1) == (wait >= 0)
            a.set_initial(prims, [0.3, 0.6])
            a.set_target(np.full(n, 8.9), np.zeros(n))
            out = []
            for _ in range(2):
                out += [[a.forward()], *a.backward(), a.final_state()]
            assert (a.team() > 0) == (wait > 0)
            return out

    ref = run(-1)
    for wait in (0, WAIT):
        for x, y in zip(run(wait), ref):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("graph", [True, False])
def test_batch_adjoint(graph):
    print(f"[fallback] batch adjoint graph={graph}", flush=True)
    cells = [3, 250, 700, 5000]
    rng = np.random.default_rng(5)
    prims = [phase_prims_to_adjoint(random_phase_prims(rng, EOS, 2)) for _ in cells]

    def run(wait):
        with BatchAdjoint([EOS] * len(cells), cells, 60, every=20) as b:
            b.set_launch(graph)
            assert (b.team(wait) > 1) == (wait >= 0)
            b.set_initial(prims, [[0.5]] * len(cells))
            b.set_target(np.full(sum(cells), 8.9), np.zeros(sum(cells)))
            out = []
            for _ in range(2):
                out += [b.forward(), *[x for g in b.backward() for x in g], b.final_state()]
            assert (b.team() > 0) == (wait > 0)
            return out

    ref = run(-1)
    for wait in (0, WAIT):
        for x, y in zip(run(wait), ref):
            assert np.array_equal(x, y)
