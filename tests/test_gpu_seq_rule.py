"""Where the sequential samplers leave their speculative batches (spec_pays,
kBatchPays): chains that take their trials singly and launches of more chains
than are resident at once give the same results, and neither costs more than
a run that never left them would show."""
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


def _chains(hip, count, lat, n, S, R):
    from brawl_amd import workloads
    v = _v(S, R)
    rng = np.random.default_rng(3)
    cfg = workloads.random_config(lat, n, workloads.equal_counts(workloads.n_atoms_of(lat, n), S), rng)
    out = []
    for k in range(count):
        L = hip.Lattice(lat, n, v)
        L.set_config(cfg)
        L.seed(50 + k)
        out.append(L)
    return out


@pytest.mark.parametrize("lat,n,S,R", [(1, (3, 3, 3), 5, 4), (2, (4, 4, 4), 2, 1)])
def test_more_chains_than_resident(hip, lat, n, S, R):
    from brawl_amd.lattice import mc_steps_batch
    from brawl_amd.nested_sampling import nested_sampling_batch
    count = 2000 if R == 1 else 600
    Ls = _chains(hip, count, lat, n, S, R)
    acc, e, _ = mc_steps_batch(Ls, [hip.beta_of(2000.0)] * count, 300, sample_every=100)
    alone = {}
    for k in (0, 1, count // 2, count - 1):
        alone[k], = _chains(hip, 1, lat, n, S, R)
        alone[k].seed(50 + k)
        a, ea = alone[k].mc_steps(hip.beta_of(2000.0), 300, sample_every=100)
        assert a == acc[k] and np.array_equal(ea, e[k])
        assert np.array_equal(alone[k].get_config(), Ls[k].get_config())
        assert all(np.array_equal(x, y) for x, y in zip(alone[k].genrand_state(), Ls[k].genrand_state()))
    p = dict(n_walkers=4, n_steps=20, n_iter=5, concentrations=np.full(S, 1.0 / S))
    res, _ = nested_sampling_batch(Ls, [p] * count)
    for k in alone:
        one, _ = nested_sampling_batch([alone[k]], [p])
        assert np.array_equal(one[0][0], res[k][0])
        assert all(np.array_equal(x, y) for x, y in zip(alone[k].genrand_state(), Ls[k].genrand_state()))
    for L in Ls + list(alone.values()):
        L.close()


def test_many_chains_do_not_take_turns(hip):
    """1024 chains of 4 shells: 7 times as long as 256 in batches alone, which
    one CU holds one chain of; about the same time one trial at a time."""
    from brawl_amd.lattice import mc_steps_batch
    Ls = _chains(hip, 1024, 1, (6, 6, 6), 4, 4)
    beta = hip.beta_of(2000.0)

    def kernel_ms(count):
        return min(mc_steps_batch(Ls[:count], [beta] * count, 1000)[2] for _ in range(3))

    few, many = kernel_ms(256), kernel_ms(1024)
    print(f"256 chains {few:.2f} ms, 1024 chains {many:.2f} ms")
    for L in Ls:
        L.close()
    assert many < 2.5 * few


def test_more_walkers_than_resident(hip):
    """Wang-Landau walkers of a launch taken one trial at a time against the
    same walkers a few at a time, which take theirs in batches."""
    from brawl_amd import workloads
    from brawl_amd.wang_landau import WangLandau
    n, S, R = (3, 3, 3), 5, 4
    p = dict(bins=24, num_windows=1, bin_overlap=0.1, energy_min=-12.0, energy_max=12.0, mc_sweeps=2)
    cfg = workloads.random_config(1, n, workloads.equal_counts(108, S), np.random.default_rng(2))

    def run(walkers, first):
        with WangLandau(1, n, _v(S, R), walkers_per_window=walkers, rank_offset=first, **p) as w:
            for k in range(walkers):
                w.set_walker(k, cfg)
            acc, _ = w.sweeps(0.01, average=False)
            return acc, *w.lng_hist(), [w.get_walker(k) for k in (0, walkers - 1)]

    acc, lng, hist, ends = run(1500, 7)
    for first in (0, 1496):
        a, g, h, e = run(4, 7 + first)
        assert np.array_equal(a, acc[first:first + 4]) and a.sum() > 0
        assert np.array_equal(g, lng[first:first + 4]) and np.array_equal(h, hist[first:first + 4])
        assert np.array_equal(e[0], ends[0]) if first == 0 else np.array_equal(e[1], ends[1])
