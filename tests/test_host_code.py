"""The library's host code without a GPU: libhes.so over a stand-in for the HIP
runtime (fake_hip.cpp) in a process of its own, which plans routes, allocates
and moves states; no kernel of the scheme runs."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_device_cap.argtypes = fake.fake_device_fail_from.argtypes = [ctypes.c_size_t]
fake.fake_host_fail_from.argtypes = [ctypes.c_size_t, ctypes.c_longlong]
fake.fake_device_used.restype = ctypes.c_size_t
fake.fake_launches.restype = ctypes.c_longlong
NONE = 2 ** 64 - 1  # no limit
import numpy as np
from hyperelasticsolver_amd._lib import HesError
from hyperelasticsolver_amd.EquationsOfState import Barton2009
from hyperelasticsolver_amd.adjoint import Adjoint, BatchAdjoint
from hyperelasticsolver_amd.batched import Batch
from hyperelasticsolver_amd.solver import Solver
EOS = Barton2009()
GENERAL = Barton2009(_beta=3.577, _gamma=2.088)
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so], check=True)

    def run(script):
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(root=ROOT, so=so) + textwrap.dedent(script)],
                           cwd=ROOT, capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]

    return run


def test_route_of_a_batch(host):
    """One launch for all steps where it is measured to pay, else a launch per
    step: many problems of a few cells fill one wave of a workgroup's four."""
    host("""
    def team(P, n, flux="rusanov", eos=EOS):
        with Batch([eos] * P, [n] * P, flux=flux) as b:
            return b.team()
    for n in (3, 32, 62):
        assert team(16384, n) == team(16384, n, "hll") == team(16384, n, eos=GENERAL) == 0, n
    assert team(4096, 3) == team(4096, 32, "hll") == team(16384, 100, "hll") == 0
    assert team(16384, 124, "hll", GENERAL) == 0
    # the chip is not full, or the waves have work
    assert team(256, 3) == team(256, 3, "hll") == 256 and team(768, 3, "hll", GENERAL) == 768
    assert team(16384, 124) == team(16384, 186, "hll") == team(16384, 250, "hll", GENERAL) == 16384
    assert team(4096, 434) == 4096 and team(4096, 980, "hll") == 3 * 4096
    with BatchAdjoint([EOS] * 8192, [40] * 8192, 4) as b:
        assert b.team() == 0
    with BatchAdjoint([EOS] * 200, [40] * 200, 4) as b:
        assert b.team() == 200
    """)


def test_long_batches_take_several_launches(host):
    """The workgroups of a team next in line wait for an earlier team's last
    step: no launch takes so many steps that this could pass for a team that
    does not meet."""
    host("""
    with Batch([EOS] * 2000, [980] * 2000) as b:
        b.set_state(np.ones((14, b.N), order="F"))
        b.run(40000)
        assert fake.fake_launches(b"k_batch_resident_end") == 3
    cells, steps = [700, 20], 40000
    with BatchAdjoint([EOS] * 2, cells, steps, every=1000) as b:
        b.set_initial([np.ones((13, 1))] * 2, [[], []])
        b.set_target(np.zeros(720), np.zeros(720))
        b.forward()
        assert fake.fake_launches(b"k_badj_resident") == 3
    """)


def test_which_launches_run_together(tmp_path):
    """Launches whose workgroups wait for one another and launches that only
    hold compute units for long: who may enter beside whom, and in which order."""
    exe = str(tmp_path / "units")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread",
                    "-I" + os.path.join(ROOT, "hyperelasticsolver_amd", "csrc"),
                    os.path.join(ROOT, "tests", "units_host.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_no_exception_leaves_a_call(host):
    """Calls on a handle and point-wise calls work, or report an error, when host
    memory is short: nothing is thrown across the C interface."""
    host("""
    from hyperelasticsolver_amd.initial import prim2cons
    n = 120000  # a download shared by threads
    q = np.asfortranarray(np.arange(14.0 * n).reshape(14, n, order="F"))
    out = np.empty_like(q)
    with Solver(EOS, n) as s, Solver(EOS, 300000) as t, Batch([EOS] * 2, [900] * 2) as b:
        t.set_state(np.ones((14, 300000), order="F"))
        b.set_state(np.ones((14, 1800), order="F"))
        fake.fake_new_fails(1)
        s.set_state(q)
        got = s.get_state()
        prim2cons(EOS, q[:, :3])
        s.run(steps=4)
        t.run(steps=4)
        b.run(4)
        fake.fake_new_fails(0)
        assert np.array_equal(got, q)
    """)


def test_state_comes_back_without_page_locked_pieces(host):
    """A large state's download takes page-locked memory for every thread: with
    some of it, or none, the state still comes back."""
    host("""
    n = 120000  # 13 MB: several pieces
    q = np.asfortranarray(np.arange(14.0 * n).reshape(14, n, order="F"))
    for allowed in (0, 1, 3, 10 ** 6):
        fake.fake_host_fail_from(1 << 20, allowed)
        with Solver(EOS, n) as s:
            s.set_state(q)
            assert np.array_equal(s.get_state(), q), allowed
            assert np.array_equal(s.get_state(), q), allowed
    """)


def test_kept_memory_is_given_back_when_it_is_short(host):
    """Device memory that finished calls left for the next ones does not make a
    later allocation fail."""
    host("""
    q = np.ones((14, 100000), order="F")
    with Solver(EOS, 100000) as s:
        s.set_state(q)
    kept = fake.fake_device_used()
    assert 0 < kept <= 4 * 96 << 20
    for make in (lambda: Solver(EOS, 50000), lambda: Batch([EOS], [50000]), lambda: Adjoint(EOS, 50000, 4),
                 lambda: BatchAdjoint([EOS], [50000], 4)):
        with make():  # its size
            need = fake.fake_device_used() - kept
        fake.fake_device_cap(need + kept // 2)
        make().close()
        assert fake.fake_device_used() < kept
        fake.fake_device_cap(NONE)
        with Solver(EOS, 100000) as s:
            s.set_state(q)
        assert fake.fake_device_used() == kept
    fake.fake_device_cap(kept + 1000)
    try:
        Solver(EOS, 100000)
        assert False
    except HesError as e:
        assert "out of memory" in str(e)
    """)


def test_no_room_for_the_messages_of_a_team(host):
    """The buffers of a one-launch time loop can be done without: a handle that
    has room for everything else is created and takes a launch per step."""
    host("""
    n = 300000
    for make in (lambda: Solver(EOS, n), lambda: Solver((EOS, EOS), 20000, flux="hll"),
                 lambda: Batch([EOS] * 40, [5000] * 40), lambda: Adjoint(EOS, n, 4, every=2),
                 lambda: BatchAdjoint([EOS] * 40, [5000] * 40, 4, every=2)):
        fake.fake_device_cap(NONE)
        with make() as h:
            assert h.team() > 0
            size = fake.fake_device_used()
        assert fake.fake_device_used() == 0
        fake.fake_device_cap(size - 1000)
        with make() as h:
            assert h.team() == 0 and h.team(1000) == 0
        assert fake.fake_device_used() == 0
    """)
