"""Divided chains (bwl_metro_split.hip), beyond single short calls: that they
were divided at all, that a chain given up is made good, runs long enough for
the tags of the swaps' records to come around and for every temperature step's
slot to be used again, and radial densities summed over several samples."""
import ctypes as C

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


def _lattice(lat, n, S, R, seed=7):
    from brawl_amd import Lattice, workloads
    v = workloads.random_v(S, [25.0 / k for k in range(1, R + 1)], seed)
    L = Lattice(lat, n, v)
    rng = np.random.default_rng(seed)
    L.set_config(workloads.random_config(lat, n, workloads.dirichlet_counts(L.n_atoms, S, rng), rng))
    return L


def _ran(lib, L):
    """[workgroups, given up, one site per lane] of the last anneal."""
    out = (C.c_int32 * 3)()
    lib.bwl_test_anneal_ran(L._h, out)
    return list(out)


def _give_up(lib, L, on):
    lib.bwl_test_give_up(L._h, int(on))


def _same(a, b, A, B):
    assert np.array_equal(a.energies_of_T, b.energies_of_T) and np.array_equal(a.C_of_T, b.C_of_T)
    assert np.array_equal(a.acceptance_of_T, b.acceptance_of_T)
    assert (a.trials, a.accepted, a.e_drift_abs, a.e_drift_rel) == (b.trials, b.accepted, b.e_drift_abs, b.e_drift_rel)
    assert (a.rho_of_T is None) == (b.rho_of_T is None)
    if a.rho_of_T is not None:
        assert np.array_equal(a.rho_of_T, b.rho_of_T)
    assert np.array_equal(A.get_config(), B.get_config())


@pytest.mark.parametrize("lat,n,S,R,parts", [(2, (32, 32, 32), 4, 4, 16), (1, (24, 24, 24), 2, 3, 7), (1, (18, 18, 18), 7, 4, 3),
                                             (1, (19, 19, 19), 5, 3, 4)])
def test_divided_and_made_good(lib, lat, n, S, R, parts):
    """Whole, given up on arrival, and whole again from where that left off."""
    print("case", lat, n, S, R, flush=True)
    A, B = _lattice(lat, n, S, R), _lattice(lat, n, S, R)
    with A, B:
        for given_up in (False, True, False):
            p = dict(T=900.0, delta_T=-100.0, T_steps=2, n_sweeps=3, burn_in_sweeps=1, seed=5)
            _give_up(lib, A, given_up)
            _give_up(lib, B, False)
            a, b = A.metropolis_simulated_annealing(**p), B.metropolis_simulated_annealing(**p)
            assert _ran(lib, A)[:2] == ([1, 1] if given_up else [parts, 0])
            assert _ran(lib, B)[:2] == [parts, 0]
            _same(a, b, A, B)


def test_given_up_in_a_batch(lib):
    from brawl_amd import anneal_batch
    shapes = [(1, (24, 24, 24), 3, 3), (2, (28, 28, 28), 4, 4), (1, (8, 8, 8), 2, 2), (2, (32, 32, 32), 4, 4)]
    A, B = [_lattice(*s) for s in shapes], [_lattice(*s) for s in shapes]
    ps = [dict(T=800.0 + 50 * k, n_sweeps=3, seed=5 + k) for k in range(len(shapes))]
    _give_up(lib, A[1], True)
    a, b = anneal_batch(A, ps)[0], anneal_batch(B, ps)[0]
    assert [_ran(lib, L)[1] for L in A] == [0, 1, 0, 0] and not any(_ran(lib, L)[1] for L in B)
    assert _ran(lib, B[1])[0] > 1 and _ran(lib, B[3])[0] > 1
    for k in range(len(shapes)):
        _same(a[k], b[k], A[k], B[k])
    for L in A + B:
        L.close()


@pytest.mark.parametrize("lat,n,S,R,chains,divided", [(2, (30, 30, 30), 3, 2, 9, 9), (1, (22, 22, 22), 4, 3, 26, 26),
                                                      (1, (18, 18, 18), 4, 4, 40, 40)])
def test_batch_is_divided(lib, lat, n, S, R, chains, divided):
    """Every chain of the batches that are compared with undivided ones."""
    from brawl_amd import anneal_batch
    A = [_lattice(lat, n, S, R, 31 + k) for k in range(chains)]
    anneal_batch(A, [dict(T=900.0, n_sweeps=1, seed=k) for k in range(chains)])
    ran = [_ran(lib, L) for L in A]
    print(ran)
    assert sum(r[0] > 1 for r in ran) == divided and not any(r[1] for r in ran)
    for L in A:
        L.close()


def test_more_rounds_than_tags(lib):
    """Rounds (of at most 384 pairs) beyond 65,536: records are cleared at 32768
    and their tags come around at 65536; three temperature steps use the first
    one's slot again."""
    A, B = _lattice(1, (18, 18, 18), 3, 3), _lattice(1, (18, 18, 18), 3, 3)
    with A, B:
        p = dict(T=1200.0, delta_T=-300.0, T_steps=3, n_sweeps=360, burn_in_sweeps=10, seed=5, asro_every=7)
        a = A.metropolis_simulated_annealing(**p)
        assert _ran(lib, A)[0] > 1 and _ran(lib, A)[1] == 0
        _give_up(lib, B, True)
        b = B.metropolis_simulated_annealing(**p)
        assert _ran(lib, B)[:2] == [1, 1]
        assert a.trials > 384 * 65536
        _same(a, b, A, B)


@pytest.mark.parametrize("lat,n,S,R,every", [(2, (24, 24, 24), 3, 4, 2), (1, (18, 18, 18), 5, 3, 3), (2, (30, 30, 30), 6, 2, 1)])
def test_radial_densities_of_several_samples(lib, lat, n, S, R, every):
    A, B = _lattice(lat, n, S, R), _lattice(lat, n, S, R)
    with A, B:
        p = dict(T=900.0, delta_T=-150.0, T_steps=3, n_sweeps=7, burn_in_sweeps=2, seed=9, asro_every=every)
        a = A.metropolis_simulated_annealing(**p)
        assert _ran(lib, A)[0] > 1 and _ran(lib, A)[1] == 0
        _give_up(lib, B, True)
        b = B.metropolis_simulated_annealing(**p)
        assert _ran(lib, B)[:2] == [1, 1]
        _same(a, b, A, B)


def test_which_small_chains_run_one_site_per_lane(lib):
    from brawl_amd import anneal_batch
    with _lattice(1, (9, 9, 9), 5, 2) as small, _lattice(1, (20, 20, 20), 5, 2) as big:
        p = dict(T=900.0, n_sweeps=2, seed=1)
        small.metropolis_simulated_annealing(**p)
        assert _ran(lib, small) == [1, 0, 1]
        anneal_batch([small, big], [p, dict(p, seed=2)])
        assert _ran(lib, small)[2] == 0 and _ran(lib, big)[2] == 0


@pytest.mark.parametrize("lat,n,S,R,sweeps,divided", [
    (1, 17, 3, 4, 40, False), (1, 18, 3, 4, 40, True),      # small enough for one site per lane in one workgroup
    (1, 19, 7, 3, 40, False), (1, 20, 7, 3, 40, True),      # 64-bit counts
    (2, 19, 6, 4, 40, False), (1, 18, 6, 4, 40, True),
    (2, 18, 2, 1, 2, False), (2, 18, 2, 1, 40, True),       # one shell: short runs are not
])
def test_which_chains_are_divided(lib, lat, n, S, R, sweeps, divided):
    """Each side of the rule's lines."""
    with _lattice(lat, (n, n, n), S, R) as L:
        L.metropolis_simulated_annealing(T=900.0, n_sweeps=sweeps, seed=1)
        assert (_ran(lib, L)[0] > 1) == divided and _ran(lib, L)[1] == 0
