"""Counts, site energies and configurations of boxes at the edges of the
measuring kernels: boxes shorter than the halo (whose planes wrap onto
themselves), one plane of cells, rows that end inside an 8-cell access, every
number of shells of both lattices, and more planes than sites in a block."""
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


CASES = [(1, (1, 1, 1), 2, 6), (2, (1, 1, 1), 2, 10), (1, (1, 3, 1), 3, 4), (2, (3, 1, 2), 8, 10), (1, (2, 5, 40), 2, 1),
         (2, (5, 3, 33), 4, 3), (1, (9, 17, 1), 5, 5), (2, (23, 13, 3), 3, 7), (1, (11, 7, 5), 8, 2)]


@pytest.mark.parametrize("lat,n,S,R", CASES)
def test_counts_energies_configuration(hip, oracle, lat, n, S, R):
    from brawl_amd import workloads
    print("case", lat, n, S, R, flush=True)
    v = workloads.random_v(S, [20.0 / k for k in range(1, R + 1)], 3 + R)
    ref = oracle.OracleLattice(lat, n, v)
    gen = oracle.Generator(5)
    cfg = ref.initial_setup(gen, concentrations=np.full(S, 1.0 / S))
    with hip.Lattice(lat, n, v) as L:
        L.set_config(cfg)
        assert np.array_equal(L.get_config(), cfg)
        h = L.pair_histogram()
        assert np.array_equal(h, ref.histogram(cfg))
        assert L.total_energy() == ref.energy_from_histogram(h)
        for _ in range(5):
            a, b = ref.random_site(gen), ref.random_site(gen)
            assert L.nbr_energy(1, *a) == ref.site_energy(cfg, *a)
            assert L.pair_energy((1,) + a, (1,) + b) == ref.pair_energy(cfg, a, b)
