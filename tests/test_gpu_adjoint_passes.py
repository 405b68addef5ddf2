"""The adjoint's first pass in one launch and its recompute of whole segments,
at the edges of their workgroups: the forward pass against a launch per step, and
gradients with the states between checkpoints recomputed against gradients with
every state kept, bit for bit (the same arithmetic).  Only where the batched
solver's states stand beside the adjoint's, whose initial states another routine
forms, is there a tolerance."""
import numpy as np
import pytest

from hyperelasticsolver_amd.EquationsOfState import Barton2009
from hyperelasticsolver_amd.adjoint import Adjoint, BatchAdjoint, phase_prims_to_adjoint
from hyperelasticsolver_amd.batched import Batch
from hyperelasticsolver_amd.initial import prim2cons, random_interfaces, random_phase_prims

pytestmark = pytest.mark.gpu

# one workgroup of the recompute and several (498 cells alone, 448 each; 250 and
# 200 in the last sizes), the first pass's workgroup shapes, both sides of the size from which only states
# near a cotangent are recomputed (on 256 compute units), and a first pass
# step by step
SIZES = [3, 250, 251, 498, 499, 896, 897, 1000, 59905, 47616, 47617, 123393, 250369, 377345]
STEPS = 53  # two full launches of the recompute and a part of one


def _problem(n):
    rng = np.random.default_rng(n)
    eos = Barton2009()
    k = 5 if n > 60 else 2
    prims14 = random_phase_prims(rng, eos, k)
    ifc = random_interfaces(rng, k - 1)
    return eos, prims14, phase_prims_to_adjoint(prims14), list(ifc)


@pytest.mark.parametrize("n", SIZES)
def test_first_pass_equals_stepwise(n):
    print(f"[adjoint passes] forward n={n}", flush=True)
    eos, prims14, prims, ifc = _problem(n)
    zero = np.zeros(n)
    with Adjoint(eos, n, STEPS, every=20) as a:
        a.set_initial(prims, ifc)
        a.set_target(zero, zero)
        loss = a.forward()
        q = a.final_state()
        assert a.forward() == loss
        assert np.array_equal(q, a.final_state())
        assert (a.team() > 0) == (n < 377345) and a.team(-1) == 0
        assert a.forward() == loss
        assert np.array_equal(q, a.final_state())
    with Batch([eos], [n], flux="rusanov") as b:
        b.set_piecewise([prim2cons(eos, prims14)], [ifc])
        b.run(STEPS, mode="eager")
        r = b.get_state()
    # the initial states come from two routines that may differ in the last
    # bits, which 53 steps carry along
    scale = np.abs(r).max(axis=1, keepdims=True) + 1e-300
    assert np.all(np.abs(q - r) <= 1e-10 * scale)


@pytest.mark.parametrize("n", SIZES)
def test_recomputed_states_change_nothing(n):
    print(f"[adjoint passes] gradients n={n}", flush=True)
    eos, _, prims, ifc = _problem(n)
    # a misfit on a few cells, so that most tiles stay without a cotangent
    with Adjoint(eos, n, STEPS, every=STEPS) as a:
        a.set_initial(prims, ifc)
        a.set_target(np.zeros(n), np.zeros(n))
        a.forward()
        rho, u = a.profiles()
    rho = rho.copy()
    rho[n // 3:n // 3 + 5] *= 1.01

    def gradient(every, sparse, graph=True):
        with Adjoint(eos, n, STEPS, every=every) as a:
            a.set_sparse(sparse)
            a.set_launch(graph)
            a.set_initial(prims, ifc)
            a.set_target(rho, u)
            out = []
            for _ in range(2):  # a captured pass replays
                loss = a.forward()
                g, gm = a.backward()
                out.append(np.concatenate([[loss], g.ravel(), gm]))
            assert np.array_equal(out[0], out[1])
            return out[0]

    ref = gradient(1, False)
    assert np.all(np.isfinite(ref)) and np.abs(ref).max() > 0.0
    for every, sparse, graph in ((2, True, True), (26, False, True), (27, True, True),
                                 (STEPS, True, False), (STEPS, False, True)):
        assert np.array_equal(gradient(every, sparse, graph), ref), (every, sparse)


# few workgroups (a tile per wave), more than the chip holds at once (two), a
# problem that does not fit and runs step by step; then the lengths that a
# workgroup of the recompute holds (126 cells alone, 122 each; with longer
# problems 250 and 244), one more, and waves past a problem's end (its last cell
# in a wave's first or last lane)
BATCHES = [[3, 62, 250, 251, 498, 499, 896, 897, 1000, 9000], [8000] * 40 + [5, 700], [123393, 300],
           [3, 62, 63, 64], [3, 65, 125, 126], [123, 124, 127, 128, 129, 183, 184, 185], [243, 244, 245, 247],
           [20] * 30 + [365, 366, 367, 2000], [1000, 1001, 1200, 1452, 1453, 251, 250, 249, 5000]]


@pytest.mark.parametrize("which", range(len(BATCHES)))
def test_batch_passes(which):
    """Forward states and gradients of a batch: the one-problem adjoint's
    states to the bit, and the same gradients whatever is recomputed."""
    cells = BATCHES[which]
    print(f"[adjoint passes] batch of {len(cells)}, up to {max(cells)} cells", flush=True)
    rng = np.random.default_rng(which)
    eos = [Barton2009(_rho0=8.93 * x, _b0=2.1 * y) for x, y in rng.uniform(0.9, 1.1, (len(cells), 2))]
    prims = [phase_prims_to_adjoint(random_phase_prims(rng, e, 2)) for e in eos]
    ifc = [[0.5]] * len(cells)
    off = np.concatenate([[0], np.cumsum(cells)])
    zero = np.zeros(off[-1])

    def run(every, sparse, graph=True, target=None):
        with BatchAdjoint(eos, cells, STEPS, every=every) as b:
            b.set_sparse(sparse)
            b.set_launch(graph)
            b.set_initial(prims, ifc)
            b.set_target(*(target or (zero, zero)))
            out = []
            for _ in range(2):
                loss = b.forward()
                out.append(np.concatenate([np.ravel(loss)] + [np.ravel(x) for g in b.backward() for x in g]))
            assert np.array_equal(out[0], out[1])
            return out[0], b.final_state(), b.profiles()

    _, state, (rho, u) = run(STEPS, True)
    for p in {0, len(cells) // 2, len(cells) - 1}:
        n, sl = cells[p], slice(off[p], off[p + 1])
        with Adjoint(eos[p], n, STEPS, every=STEPS) as a:
            a.set_initial(prims[p], ifc[p])
            a.set_target(zero[sl], zero[sl])
            a.forward()
            assert np.array_equal(a.final_state(), state[:, sl]), p
    rho = rho.copy()
    rho[off[:-1] + np.array(cells) // 3] *= 1.01  # one observed cell per problem
    u = u.copy()
    u[off[1:] - 1 - (np.array(cells) > 9)] += 0.01  # and one at its end
    ref = run(1, False, target=(rho, u))[0]
    assert np.all(np.isfinite(ref)) and np.abs(ref).max() > 0.0
    for every, sparse, graph in ((2, True, True), (26, False, True), (27, True, False), (STEPS, True, True)):
        assert np.array_equal(run(every, sparse, graph, (rho, u))[0], ref), (every, sparse, graph)


@pytest.mark.parametrize("every", [4096, 5000])  # a checkpoint where two launches meet, and none
def test_batch_first_pass_in_two_launches(every):
    """More steps than one launch of the first pass takes: the losses, states
    and gradients of a launch per step."""
    cells, steps = [300, 20, 3], 16384 + 50
    print(f"[adjoint passes] batch, {steps} steps, every {every}", flush=True)
    eos = [Barton2009()] * len(cells)
    rng = np.random.default_rng(every)
    prims = [phase_prims_to_adjoint(random_phase_prims(rng, e, 2)) for e in eos]

    def run(wait):
        with BatchAdjoint(eos, cells, steps, every=every) as b:
            b.team(wait)
            b.set_initial(prims, [[0.5]] * len(cells))
            b.set_target(np.full(sum(cells), 8.9), np.zeros(sum(cells)))
            losses = b.forward()
            out = [losses, b.final_state()] + [x for g in b.backward() for x in g]
            assert (b.team() > 0) == (wait > 0)
            return out

    ref = run(-1)
    assert np.all(np.isfinite(ref[0])) and np.all(np.isfinite(ref[1]))
    for x, y in zip(run(4_000_000), ref):
        assert np.array_equal(x, y, equal_nan=True)
