"""Small chains at one site per lane (bwl_metro_alone.hip) against the kernel
with one pair per lane, bit for bit: the same chain alone and in a batch with
a chain too large for it, which keeps both on the other kernel.  One to four
rows of pairs, a round smaller than half a row, both lattices, the three count
words, burn-in, two temperatures."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import brawl_amd
    from brawl_amd import _lib
    _lib.load()
    if _lib.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return brawl_amd


def _lattice(hip, lat, n, S, R):
    from brawl_amd import workloads
    v = workloads.random_v(S, [30.0 / k for k in range(1, R + 1)], 3)
    L = hip.Lattice(lat, (n, n, n), v)
    L.seed(7 + n)
    L.initial_setup(species_numbers=workloads.equal_counts(L.n_atoms, S))
    return L


@pytest.mark.parametrize("lat,n,S", [(1, 6, 2), (1, 9, 5), (1, 12, 4), (1, 16, 3), (1, 11, 6), (2, 6, 4), (2, 8, 6),
                                     (2, 13, 5), (2, 16, 2)])
def test_same_chain_as_one_pair_per_lane(hip, lat, n, S):
    print("case", lat, n, S, flush=True)
    p = dict(T=900.0, delta_T=-80.0, T_steps=2, n_sweeps=12, burn_in_sweeps=2, seed=5)
    big = _lattice(hip, lat, 20, S, 2)
    one, two = _lattice(hip, lat, n, S, 2), _lattice(hip, lat, n, S, 2)
    with big, one, two:
        alone = one.metropolis_simulated_annealing(**p)
        batch, _ = hip.anneal_batch([two, big], [p, dict(p, seed=6)])
        assert np.array_equal(alone.energies_of_T, batch[0].energies_of_T)
        assert np.array_equal(alone.C_of_T, batch[0].C_of_T)
        assert np.array_equal(alone.acceptance_of_T, batch[0].acceptance_of_T)
        assert (alone.trials, alone.accepted) == (batch[0].trials, batch[0].accepted)
        assert np.array_equal(one.get_config(), two.get_config())
