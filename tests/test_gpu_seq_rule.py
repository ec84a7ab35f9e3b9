"""Where the sequential sampler leaves its speculative batches (kBatchPays):
chains that take their trials singly give the same results, and boxes whose
batches are cut short no longer pay for whole ones."""
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


def _v(S, R):
    from brawl_amd import workloads
    return workloads.random_v(S, [30.0 / k for k in range(1, R + 1)], 11 * S + R)


@pytest.mark.parametrize("nbr_swap", [False, True])
@pytest.mark.parametrize("lat,n,S,R", [(1, (3, 3, 3), 5, 4), (1, (4, 3, 5), 3, 3), (1, (3, 3, 3), 8, 2), (2, (4, 4, 4), 4, 4),
                                       (2, (3, 5, 3), 3, 3), (2, (3, 3, 3), 2, 2)])
def test_nearly_all_accepted(hip, oracle, lat, n, S, R, nbr_swap):
    """Batches cut short: most trials are taken singly, with a batch tried in
    between; sampled unevenly, and a second call in the middle of the stream."""
    from brawl_amd import workloads
    print("case", lat, n, S, R, nbr_swap, flush=True)
    v = _v(S, R)
    ref = oracle.OracleLattice(lat, n, v)
    gen = oracle.Generator(77)
    cfg = ref.initial_setup(gen, species_numbers=workloads.equal_counts(ref.n_atoms, S))
    beta = hip.beta_of(30000.0)
    with hip.Lattice(lat, n, v) as L:
        L.set_config(cfg)
        L.set_genrand_state(*gen.state_arrays())
        for trials, every in ((1200, 0), (700, 13)):
            acc, energies = L.mc_steps(beta, trials, nbr_swap=nbr_swap, sample_every=every)
            acc_ref, e_ref = 0, []
            for t in range(1, trials + 1):
                acc_ref += ref.mc_step(cfg, beta, gen, nbr_swap=nbr_swap)
                if every and t % every == 0:
                    e_ref.append(ref.total_energy(cfg))
            assert acc == acc_ref
            assert energies is None or np.array_equal(energies, e_ref)
            assert np.array_equal(L.get_config(), cfg)
            mt, mti = L.genrand_state()
            mt_ref, mti_ref = gen.state_arrays()
            assert mti == mti_ref and np.array_equal(mt, mt_ref)


def test_short_batches_are_given_up(hip):
    """fcc 3^3, 4 shells, nearly all accepted, nearly every batch cut after
    one trial: 6.3 times as long as at low acceptance in batches alone."""
    import time
    from brawl_amd import workloads
    with hip.Lattice(1, (3, 3, 3), _v(5, 4)) as L:
        L.seed(3)
        L.set_config(workloads.random_config(1, (3, 3, 3), workloads.equal_counts(L.n_atoms, 5), np.random.default_rng(1)))

        def seconds(temp):
            best = np.inf
            for _ in range(4):
                t = time.perf_counter()
                L.mc_steps(hip.beta_of(temp), 20000)
                best = min(best, time.perf_counter() - t)
            return best

        low, high = seconds(300.0), seconds(1e6)
    print(f"300 K {low * 1e3:.2f} ms, 10^6 K {high * 1e3:.2f} ms")
    assert high < 4.0 * low


def test_energies_of_small_boxes(hip):
    """512 runs of 8 walkers that make one trial: 0.136 ms while each
    workgroup also built the table of list positions, 0.063 without."""
    from brawl_amd.nested_sampling import nested_sampling_batch
    Ls = [hip.Lattice(2, (4, 4, 4), _v(3, 4)) for _ in range(512)]
    p = dict(n_walkers=8, n_steps=1, n_iter=1, concentrations=np.array([0.3, 0.3, 0.4]))
    ms = min(nested_sampling_batch(Ls, [p] * len(Ls))[1] for _ in range(4))
    print(f"{ms:.3f} ms")
    for L in Ls:
        L.close()
    assert ms < 0.1
