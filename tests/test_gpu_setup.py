"""Initial configurations drawn on the device (bwl_setup.hip) against the
oracle and against the rule itself: streams that run through many blocks of
624 draws, 8 species, a rule that is drawn on the host, one stream shared by
two runs, and draws that lie exactly on the bound of two species."""
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


# one species short of atoms, equal shares, one site more than a wavefront,
# and a concentration below the device's limit (one atom in 8192 sites)
CASES = [
    (1, (6, 6, 6), 5, dict(species_numbers=[173, 173, 173, 173, 172]), 130),
    (2, (5, 3, 7), 8, dict(species_numbers=[1, 2, 3, 4, 50, 50, 50, 50]), 40),
    (1, (4, 5, 3), 3, dict(concentrations=[0.5, 0.3, 0.2]), 5),
    (2, (4, 4, 4), 2, dict(species_numbers=[127, 1]), 20),
    (2, (16, 16, 16), 2, dict(concentrations=[0.99991, 0.00009]), 2),
]


@pytest.mark.parametrize("lat,n,S,sn,W", CASES)
def test_walkers_of_a_run(hip, oracle, lat, n, S, sn, W):
    from brawl_amd import nested_sampling, workloads
    v = workloads.random_v(S, [30.0, 15.0], 5)
    if "species_numbers" in sn:
        sn = dict(species_numbers=np.array(sn["species_numbers"], dtype=np.int64))
    p = dict(n_walkers=W, n_steps=3, n_iter=W // 2, **sn)
    ref = oracle.OracleLattice(lat, n, v)
    gen = oracle.Generator(4357)
    lim_ref = ref.nested_sampling(gen, **p)
    with hip.Lattice(lat, n, v) as L:
        L.seed(4357)
        lim, _ = nested_sampling.nested_sampling(L, **p)
        state = L.genrand_state()
    assert np.array_equal(lim, lim_ref)
    mt, mti = gen.state_arrays()
    assert state[1] == mti and np.array_equal(state[0], mt)


def test_a_context_given_twice(hip):
    """Both runs' walkers come from the one stream in turn."""
    from brawl_amd import nested_sampling, workloads
    v = workloads.random_v(3, [30.0, 15.0], 5)
    p = dict(n_walkers=6, n_steps=4, n_iter=5, species_numbers=np.array([90, 83, 83], dtype=np.int64))
    with hip.Lattice(1, (4, 4, 4), v) as A, hip.Lattice(1, (4, 4, 4), v) as B:
        A.seed(99)
        res, _ = nested_sampling.nested_sampling_batch([A, A], [p, p])
        B.seed(99)
        for _ in range(6):
            B.initial_setup(species_numbers=p["species_numbers"])
            mt, mti = B.genrand_state()
            gen = np.random.RandomState()
            gen.set_state(("MT19937", mt, mti))
            gen.randint(0, 2 ** 32, dtype=np.uint32)  # the draw for the energy's jitter
            _, mt, mti = gen.get_state()[:3]
            B.set_genrand_state(mt, mti)
        alone, _ = nested_sampling.nested_sampling(B, **p)
    assert np.array_equal(res[1][0], alone)


def _untemper(y):
    y ^= y >> 18
    y ^= (y << 15) & 0xefc60000
    x = y
    for _ in range(5):
        x = y ^ ((x << 7) & 0x9d2c5680)
    y = x & 0xffffffff
    x = y
    for _ in range(3):
        x = y ^ (x >> 11)
    return x & 0xffffffff


def test_draws_on_a_bound(hip):
    """Draws equal to the bound of two species place one atom, of the first
    species that has one left."""
    from brawl_amd import nested_sampling, workloads
    n, N = (4, 4, 4), 256
    v = workloads.random_v(2, [30.0], 5)
    counts = np.array([128, 128], dtype=np.int64)
    draws = np.random.default_rng(3).integers(0, 2 ** 32, size=624, dtype=np.uint64).astype(np.uint32)
    draws[[0, 1, 2, 17, 63, 64, 65, 130, 200, 290, 291, 300]] = 0x80000000
    mt = np.array([_untemper(int(d)) for d in draws], dtype=np.uint32)

    def place(at):
        room, out = [128, 128], []
        while len(out) < N:
            d = int(draws[at])
            at += 1
            for s, inside in enumerate((d <= 0x80000000, d >= 0x80000000)):
                if inside and room[s] > 0:
                    room[s] -= 1
                    out.append(s + 1)
                    break
        return np.array(out, dtype=np.int8), at

    first, at = place(0)
    second, _ = place(at + 1)
    with hip.Lattice(1, n, v) as L:
        L.set_genrand_state(mt, 0)
        cfg = L.initial_setup(species_numbers=counts)
        x, y, z = np.meshgrid(*[np.arange(8)] * 3, indexing="ij")
        sites = np.flatnonzero(((x + y + z) % 2 == 0).ravel(order="F"))
        assert np.array_equal(cfg.ravel(order="F")[sites], first)
        e1 = L.total_energy()
        flat = np.zeros(512, dtype=np.int8)
        flat[sites] = second
        L.set_config(flat.reshape((8, 8, 8), order="F"))
        e2 = L.total_energy()
        L.set_genrand_state(mt, 0)
        lim, _ = nested_sampling.nested_sampling(L, n_walkers=2, n_steps=1, n_iter=1, species_numbers=counts)
    # the limit is the larger energy and a jitter of at most 1e-8
    assert abs(lim[0] - max(e1, e2)) < 1.1e-8
