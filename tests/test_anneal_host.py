"""The host side of an anneal without a device (tests/fake_hip.cpp): what is
launched, in how many workgroups, and what has been waited for.  Each test
runs in a process of its own, which loads the fake runtime before the library."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

PRELUDE = """
import ctypes as C, os, sys
sys.path.insert(0, {root!r})
fake = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)
import numpy as np
from brawl_amd import Lattice, BrawlError, anneal_batch, workloads
LAUNCH = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_longlong, C.c_void_p)
launches = []
def record(fn, grid, block, lds, stream):
    launches.append((fn, grid, block, lds, stream))
    return 0
def on_launch(f):
    on_launch.keep = LAUNCH(f)
    fake.fake_on_launch(on_launch.keep)
def lattice(lat, n, S, R):
    v = workloads.random_v(S, [25.0 / k for k in range(1, R + 1)], 3)
    L = Lattice(lat, n, v)
    L.set_config(workloads.random_config(lat, n, workloads.equal_counts(L.n_atoms, S), np.random.default_rng(1)))
    return L
def grids(f):
    launches.clear()
    f()
    return [l[1] for l in launches]
P = dict(T=900.0, n_sweeps=50, seed=1)
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so], check=True)

    def go(body):
        code = PRELUDE.format(root=ROOT, so=so) + textwrap.dedent(body)
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr

    return go


def test_divided_only_into_cus_that_are_free(run):
    """A large anneal that starts while another call's chains are in flight
    (its launch is made from inside that call's) is divided into what they
    leave of an XCD, and is divided again once they have ended."""
    run("""
    big = lattice(2, (32, 32, 32), 4, 4)
    small = [lattice(1, (16, 16, 16), 2, 2) for _ in range(200)]
    few = small[:30]
    anneal = lambda: big.metropolis_simulated_annealing(**P)
    on_launch(record)
    alone = grids(anneal)
    # (nothing runs, so the division is given up and made good undivided)
    assert len(alone) == 2 and alone[0] == 8 * 16 and alone[1] == 1, alone

    def during(call, inner):
        seen = []
        def f(fn, grid, block, lds, stream):
            if not seen:
                seen.append(None)
                on_launch(record)
                seen[0] = grids(inner)
            return 0
        on_launch(f)
        keep = on_launch.keep
        call()
        return seen[0]

    batch = lambda chains: anneal_batch(chains, [dict(P, seed=k) for k in range(len(chains))])
    assert during(lambda: batch(small), anneal) == [1]        # 25 a CU's worth on each XCD: 7 left
    assert during(lambda: batch(few), anneal)[0] == 8 * 16     # 4 on each
    from brawl_amd.lattice import mc_steps_batch
    assert during(lambda: mc_steps_batch(small, [1.0] * 200, 10), anneal) == [1]
    assert grids(anneal)[0] == 8 * 16
    """)


def test_given_up_division_is_made_good(run):
    """The chain that did not complete is run again undivided, its results
    and those of the others are whole."""
    run("""
    lib = Lattice(1, (1, 1, 1), np.zeros((2, 2, 1)))._L
    on_launch(record)
    chains = [lattice(1, (24, 24, 24), 3, 3), lattice(1, (8, 8, 8), 2, 2)]
    got = grids(lambda: anneal_batch(chains, [P, dict(P, seed=2)]))
    assert len(got) == 3 and got[0] > 8 and got[1:] == [1, 1], got
    ran = (C.c_int32 * 3)()
    lib.bwl_test_anneal_ran(chains[0]._h, ran)
    assert list(ran)[:2] == [1, 1]
    lib.bwl_test_anneal_ran(chains[1]._h, ran)
    assert list(ran) == [1, 0, 1]
    """)


def test_error_exits_wait_for_what_was_queued(run):
    """A batch of three kernels whose first, second or third launch fails: no
    stream has work in flight once the call has returned, on which the next
    call's arguments or the context's end could come."""
    run("""
    chains = [lattice(1, (12, 12, 12), 2, 2), lattice(2, (12, 12, 12), 3, 2), lattice(1, (12, 12, 12), 3, 3)]
    params = [dict(P, seed=k) for k in range(3)]
    on_launch(record)
    assert len(grids(lambda: anneal_batch(chains, params))) == 3
    assert len({l[4] for l in launches}) == 3 and fake.fake_busy() == 0
    for which in range(3):
        count = [0]
        def fail(fn, grid, block, lds, stream):
            count[0] += 1
            return int(count[0] == which + 1)
        on_launch(fail)
        keep = on_launch.keep
        try:
            anneal_batch(chains, params)
        except BrawlError:
            pass
        else:
            raise AssertionError("no error")
        assert fake.fake_busy() == 0, (which, fake.fake_busy())
    on_launch(record)
    for L in chains:
        L.close()
    assert fake.fake_freed_busy() == 0
    """)


def test_pinned_blocks_of_a_context(run):
    """A context that takes one configuration, or large ones only, makes no
    pinned block; the blocks that it makes go with the last context."""
    run("""
    v = np.zeros((2, 2, 1))
    def cfg(n):
        return workloads.random_config(1, n, workloads.equal_counts(4 * n[0] * n[1] * n[2], 2), np.random.default_rng(1))
    small, large = (8, 8, 8), (60, 60, 60)
    for n, calls in ((small, 1), (large, 3)):
        with Lattice(1, n, v) as L:
            for _ in range(calls):
                L.set_config(cfg(n))
            if n is large:
                L.get_config()
            assert fake.fake_pinned_made() == 0
    with Lattice(1, small, v) as L, Lattice(1, small, v) as M:
        for _ in range(3):
            L.set_config(cfg(small))
            M.set_config(cfg(small))
            L.get_config()
        assert fake.fake_pinned_made() == fake.fake_pinned_held() == 1
    assert fake.fake_pinned_held() == 0
    """)
