"""The sequential samplers in speculative batches (bwl_spec.h) against the
oracle, bit for bit: the smallest boxes each shell count allows (where a swap
reaches most of a batch) and uneven ones, 2 to 8 species, and a composition
with one solute atom (whose second sites lie hundreds of draws ahead)."""
import sys

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


# lattice, n, S, R: every shell count at its smallest box (all axes longer
# than twice the range), then uneven boxes
SHAPES = [
    (1, (2, 2, 2), 2, 1), (1, (3, 3, 3), 8, 2), (1, (3, 3, 3), 3, 3), (1, (3, 3, 3), 5, 4),
    (2, (2, 2, 2), 2, 1), (2, (3, 3, 3), 4, 2), (2, (3, 3, 3), 3, 3), (2, (4, 4, 4), 7, 4),
    (1, (3, 5, 4), 2, 4), (2, (4, 7, 5), 6, 4), (2, (3, 3, 11), 2, 2),
]


def _case(hip, oracle, lat, n, S, R, solute):
    from brawl_amd import workloads
    print("case", lat, n, S, R, "one solute" if solute else "", flush=True)
    sys.stdout.flush()
    v = workloads.random_v(S, [30.0 / k for k in range(1, R + 1)], 11 * S + R)
    ref = oracle.OracleLattice(lat, n, v)
    N = ref.n_atoms
    counts = workloads.dirichlet_counts(N, S, np.random.default_rng(N))
    if solute:
        counts = np.array([N - 1] + [1] + [0] * (S - 2), dtype=np.int64)
    return v, ref, counts


def _same_state(state, gen):
    mt, mti = gen.state_arrays()
    assert state[1] == mti and np.array_equal(state[0], mt)


@pytest.mark.parametrize("lat,n,S,R,solute", [s + (False,) for s in SHAPES] + [(2, (4, 4, 4), 2, 2, True)])
def test_nested_sampling(hip, oracle, lat, n, S, R, solute):
    from brawl_amd import nested_sampling
    v, ref, counts = _case(hip, oracle, lat, n, S, R, solute)
    gen = oracle.Generator(4357)
    p = dict(n_walkers=7, n_steps=23, n_iter=60, species_numbers=counts)
    lim_ref = ref.nested_sampling(gen, **p)
    with hip.Lattice(lat, n, v) as L:
        L.seed(4357)
        lim, _ = nested_sampling.nested_sampling(L, **p)
        state = L.genrand_state()
    assert np.array_equal(lim, lim_ref)
    _same_state(state, gen)


@pytest.mark.parametrize("nbr_swap", [False, True])
@pytest.mark.parametrize("lat,n,S,R", SHAPES)
def test_wang_landau_sweeps(hip, oracle, lat, n, S, R, nbr_swap):
    """Two windows over the energies of random configurations, so that some
    walkers start inside theirs and some outside."""
    from brawl_amd import wang_landau
    v, ref, counts = _case(hip, oracle, lat, n, S, R, False)
    span = 12.0
    wl = wang_landau.WangLandau(lat, n, v, bins=24, num_windows=2, walkers_per_window=3, bin_overlap=0.1,
                                energy_min=-span, energy_max=span, mc_sweeps=3, nbr_swap=nbr_swap)
    _, edges = ref.wl_setup(24, 2, 0.1, -span, span)
    wl.initial_setup(species_numbers=counts)
    lng0 = np.random.default_rng(5).normal(0.0, 0.5, (wl.n_walkers, wl.bins))
    wl.set_lng_hist(lng0, np.zeros((wl.n_walkers, wl.hist_stride)))
    acc, _ = wl.sweeps(0.7, average=False)
    lng, hist = wl.lng_hist()
    for k in range(wl.n_walkers):
        gen = oracle.Generator(rank=k)
        cfg = ref.initial_setup(gen, species_numbers=counts)
        s, e = (int(q) for q in wl.windows[wl.window_of(k)])
        lk, h = lng0[k].copy(), np.zeros(e - s + 1)
        a = ref.wl_sweeps(cfg, gen, mc_sweeps=3, bin_edges=edges, start_idx=s, end_idx=e, wl_f=0.7, lng=lk, hist=h,
                          nbr_swap=nbr_swap)
        assert acc[k] == a
        assert np.array_equal(lng[k], lk) and np.array_equal(hist[k, :e - s + 1], h)
        assert np.array_equal(wl.get_walker(k), cfg)
        _same_state(wl.genrand_state(k), gen)
    wl.close()


@pytest.mark.parametrize("nbr_swap", [False, True])
@pytest.mark.parametrize("temp", [200.0, 3000.0])
@pytest.mark.parametrize("lat,n,S,R", SHAPES)
def test_sequential_metropolis(hip, oracle, lat, n, S, R, temp, nbr_swap):
    """Uneven sampling, so that batches end at samples and at the run's end;
    the second call starts in the middle of the stream's block."""
    v, ref, counts = _case(hip, oracle, lat, n, S, R, False)
    gen = oracle.Generator(77)
    cfg = ref.initial_setup(gen, species_numbers=counts)
    beta = hip.beta_of(temp)
    with hip.Lattice(lat, n, v) as L:
        L.set_config(cfg)
        L.set_genrand_state(*gen.state_arrays())
        for trials, every in ((1, 0), (1500, 37)):
            acc, energies = L.mc_steps(beta, trials, nbr_swap=nbr_swap, sample_every=every)
            acc_ref, e_ref = 0, []
            for t in range(1, trials + 1):
                acc_ref += ref.mc_step(cfg, beta, gen, nbr_swap=nbr_swap)
                if every and t % every == 0:
                    e_ref.append(ref.total_energy(cfg))
            assert acc == acc_ref
            assert energies is None or np.array_equal(energies, e_ref)
            assert np.array_equal(L.get_config(), cfg)
            _same_state(L.genrand_state(), gen)
