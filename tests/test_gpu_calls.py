"""Point-wise calls over their three routes: small calls in page-locked memory,
larger ones through kept device memory, and two-phase faces by groups of lanes
(up to 4096 faces) or one lane each."""
import threading

import numpy as np
import pytest

from hyperelasticsolver_amd import HyperelasticityMPh, NumFluxes
from hyperelasticsolver_amd._lib import DomainError
from hyperelasticsolver_amd.EquationsOfState import Barton2009
from hyperelasticsolver_amd.initial import prim2cons, random_two_phase_prims

pytestmark = pytest.mark.gpu

EOS = (Barton2009(), Barton2009(_rho0=2.7, _b0=3.1))
MATS = np.concatenate([e.params() for e in EOS])


def _faces(n, seed):
    """n faces cycling through 7 pairs of states, two of them without a jump."""
    rng = np.random.default_rng(seed)
    ql = prim2cons(EOS, random_two_phase_prims(rng, EOS, 7))
    qr = prim2cons(EOS, random_two_phase_prims(rng, EOS, 7))
    qr[:, 2] = ql[:, 2]
    qr[[0, 15], 4] = ql[[0, 15], 4]
    k = np.arange(n) % 7
    return ql, qr, np.asfortranarray(ql[:, k]), np.asfortranarray(qr[:, k]), k


# one face; the last of a wave of groups and the next; the last call in page-
# locked memory (108 faces of 5 x 30 values) and the next; the last by groups
# and the next
@pytest.mark.parametrize("flux", ["lxf", "hll"])
@pytest.mark.parametrize("n", [1, 4, 5, 108, 109, 4096, 4097])
def test_faces_against_the_oracle(ora, n, flux):
    print(f"[calls] faces n={n} flux={flux}", flush=True)
    pl, pr, ql, qr, k = _faces(n, n)
    el, er = (HyperelasticityMPh.get_eigvals(EOS, q, [1.0, 0.0, 0.0]) for q in (ql, qr))
    got = (NumFluxes.hll(EOS, ql, qr, (el, er)) if flux == "hll" else NumFluxes.lxf(EOS, ql, qr, 5.0))
    for j in range(min(n, 7)):
        if flux == "hll":
            ref = ora.hll(2, MATS, pl[:, j], pr[:, j], el[:, j], er[:, j])
        else:
            ref = ora.lxf(2, MATS, pl[:, j], pr[:, j], 5.0)
        for g, r in zip(got, ref):
            g = g.reshape(30, -1)
            assert np.array_equal(g[:, k == j], np.repeat(g[:, j:j + 1], (k == j).sum(), axis=1))
            # 18 quadrature nodes of O(100) operations each: 1e-12 of the largest component
            assert np.abs(g[:, j] - np.asarray(r)).max() <= 1e-12 * max(1.0, np.abs(r).max())


@pytest.mark.parametrize("n", [1, 300, 5000])
def test_bad_state_in_every_route(n):
    print(f"[calls] bad state n={n}", flush=True)
    _, _, q, _, _ = _faces(n, 3)
    good = HyperelasticityMPh.cons2prim_mph(EOS, q)
    bad = q.copy(order="F")
    bad[6:15, n - 1] *= -1.0  # det(rho A) < 0
    with pytest.raises(DomainError):
        HyperelasticityMPh.cons2prim_mph(EOS, bad)
    assert np.array_equal(HyperelasticityMPh.cons2prim_mph(EOS, q), good)


def test_calls_from_many_threads():
    sizes = [1, 9, 200, 3000]
    data = [_faces(n, n)[2] for n in sizes]
    ref = [HyperelasticityMPh.cons2prim_mph(EOS, q) for q in data]
    wrong = []

    def work(k):
        for r in range(20):
            j = (k + r) % len(sizes)
            if not np.array_equal(HyperelasticityMPh.cons2prim_mph(EOS, data[j]), ref[j]):
                wrong.append((k, r))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
