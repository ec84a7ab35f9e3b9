"""Anneals whose chains are divided over several workgroups
(bwl_metro_split.hip) against the same chains run by one workgroup each
(bwl_metropolis_anneal_noalloc, which divides none), bit for bit: energies,
specific heats, acceptances, counts and configurations.  The shapes take
every form of the division: one and two passes, rows that the parts do not
share out evenly, the smallest rounds that are divided, all three widths of
the shell counts, and batches in which some chains have fewer parts."""
import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from brawl_amd import _lib
    L = _lib.load()
    if _lib.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return L


def _lattice(lat, n, S, R, seed):
    from brawl_amd import Lattice, workloads
    v = workloads.random_v(S, [25.0 / k for k in range(1, R + 1)], seed)
    L = Lattice(lat, n, v)
    L.set_config(workloads.random_config(lat, n, workloads.dirichlet_counts(L.n_atoms, S, np.random.default_rng(seed)),
                                         np.random.default_rng(seed + 1)))
    return L


def _undivided(lib, L, p):
    from brawl_amd import _lib
    T = p.T_steps
    e, c, a = np.zeros(T), np.zeros(T), np.zeros(T)
    st = _lib.RunStats()
    dp = C.POINTER(C.c_double)
    rc = lib.bwl_metropolis_anneal_noalloc(L._h, C.byref(p), e.ctypes.data_as(dp), c.ctypes.data_as(dp),
                                           a.ctypes.data_as(dp), C.byref(st))
    assert rc == 0, lib.bwl_last_error()
    return e, c, a, st


def _check(lib, lat, n, S, R, chains, T_steps=2, n_sweeps=2, burn=1, calls=1):
    from brawl_amd import _lib, anneal_batch
    print("divided", lat, n, S, R, chains, flush=True)
    sys.stdout.flush()
    A = [_lattice(lat, n, S, R, 31 + k) for k in range(chains)]
    B = [_lattice(lat, n, S, R, 31 + k) for k in range(chains)]
    for call in range(calls):  # a second call goes on with the streams
        ps = [dict(T=900.0 + 50 * k, delta_T=-200.0, T_steps=T_steps, n_sweeps=n_sweeps, burn_in_sweeps=burn,
                   seed=5 + k) for k in range(chains)]
        res, _ = anneal_batch(A, ps)
        for k in range(chains):
            e, c, a, st = _undivided(lib, B[k], _lib.AnnealParams(ps[k]["T"], -200.0, T_steps, n_sweeps, burn, 0, 5 + k))
            r = res[k]
            assert np.array_equal(r.energies_of_T, e) and np.array_equal(r.C_of_T, c)
            assert np.array_equal(r.acceptance_of_T, a)
            assert r.trials == st.trials > 0 and r.accepted == st.accepted
            assert r.e_drift_abs == st.e_drift_abs
            assert np.array_equal(A[k].get_config(), B[k].get_config())
    for L in A + B:
        L.close()


@pytest.mark.parametrize("lat,n,S,R", [
    (2, (32, 32, 32), 4, 4),  # its own kernel, two passes, 16 parts
    (2, (30, 30, 30), 6, 2),  # two passes, 64-bit counts
    (2, (26, 26, 26), 5, 3),  # 6-bit fields
    (2, (20, 20, 20), 3, 4),  # 7 rows among 4 parts
    (2, (24, 24, 24), 8, 2),  # close to the smallest rounds divided
    (1, (24, 24, 24), 2, 3),
    (1, (17, 17, 17), 4, 4),  # odd extents
    (1, (16, 16, 16), 7, 4),
])
def test_single_chain(lib, lat, n, S, R):
    _check(lib, lat, n, S, R, 1, calls=2)


@pytest.mark.parametrize("lat,n,S,R,chains", [
    (2, (30, 30, 30), 3, 2, 9),   # 8 chains of 16 parts and one of 8
    (1, (22, 22, 22), 4, 3, 26),
    (1, (16, 16, 16), 4, 4, 40),
])
def test_batch(lib, lat, n, S, R, chains):
    _check(lib, lat, n, S, R, chains, T_steps=1, n_sweeps=1)


@pytest.mark.parametrize("lat,n,S,R", [(2, (24, 24, 24), 3, 4), (1, (16, 16, 16), 5, 4)])
def test_radial_densities(lib, lat, n, S, R):
    """One sweep, one sample: a divided chain's rho_of_T equals the radial
    densities of its final configuration."""
    with _lattice(lat, n, S, R, 7) as L:
        r = L.metropolis_simulated_annealing(T=900.0, n_sweeps=1, seed=5, asro_every=1)
        assert np.array_equal(r.rho_of_T[:, :, :, 0], L.radial_densities(R + 1))
