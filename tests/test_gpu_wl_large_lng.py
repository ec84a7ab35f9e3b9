"""Wang-Landau sweeps on a ln g so large that adding ln f rounds: the walkers'
quick decisions (k_wl_sweeps_spec) take products for sums of ln f, which is
near enough only while ln g is small."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,wl_f", [(0.0, 0.7), (4e9, 0.7), (3e12, 0.7), (-1e13, 0.7), (2e15, 0.7), (5.0, 3e11)])
def test_sweeps(oracle, level, wl_f):
    from brawl_amd import wang_landau, workloads
    print("case", level, wl_f, flush=True)
    lat, n, S, R, span, sweeps = 2, (5, 4, 4), 3, 2, 8.0, 40
    v = workloads.random_v(S, [30.0, 15.0], 5)
    ref = oracle.OracleLattice(lat, n, v)
    counts = workloads.equal_counts(ref.n_atoms, S)
    with wang_landau.WangLandau(lat, n, v, bins=24, num_windows=1, walkers_per_window=4, bin_overlap=0.1,
                                energy_min=-span, energy_max=span, mc_sweeps=sweeps) as w:
        w.initial_setup(species_numbers=counts)
        lng0 = level + np.random.default_rng(5).normal(0.0, 1.0, (w.n_walkers, w.bins))
        w.set_lng_hist(lng0, np.zeros((w.n_walkers, w.hist_stride)))
        acc, _ = w.sweeps(wl_f, average=False)
        lng, hist = w.lng_hist()
        for k in range(w.n_walkers):
            gen = oracle.Generator(rank=k)
            cfg = ref.initial_setup(gen, species_numbers=counts)
            s, e = (int(q) for q in w.windows[0])
            lk, h = lng0[k].copy(), np.zeros(e - s + 1)
            a = ref.wl_sweeps(cfg, gen, mc_sweeps=sweeps, bin_edges=w.bin_edges, start_idx=s, end_idx=e, wl_f=wl_f, lng=lk,
                              hist=h)
            assert a > 0 and acc[k] == a
            assert np.array_equal(lng[k], lk) and np.array_equal(hist[k, :e - s + 1], h)
            assert np.array_equal(w.get_walker(k), cfg)
            mt, mti = w.genrand_state(k)
            mt_ref, mti_ref = gen.state_arrays()
            assert mti == mti_ref and np.array_equal(mt, mt_ref)
