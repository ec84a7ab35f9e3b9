"""What a user of this library has it do, as measurable cases.

A case is one of the library's calls (or the few calls that a program makes
together) at one size.  `listed()` holds the sizes that stand for the use of
each call, `draw()` gives more of the same ranges.  `prepare()` makes what a
program holds before the call, `run()` makes the call, `work()` prices it and
`exact()` recomputes in numpy what can be recomputed outside the library.
"""
import functools
import math

import numpy as np

from brawl_amd import lattice as _lat
from brawl_amd import workloads as _wl

FCC, BCC = 1, 2
CODE = {"fcc": FCC, "bcc": BCC}
# squared shell distances on the doubled grid
SHELLS = {"fcc": [2, 4, 6, 8, 10, 12], "bcc": [3, 4, 8, 11, 12, 16, 19, 20, 24, 27]}


def listed():
    return [
        # The Hamiltonian's pair energy of two sites of a lattice held on the
        # device: the smallest call, made by hosts that keep their own trial
        # loop (binary fcc 8^3, two shells: the serial example).
        dict(name="pair_energy", kind="pair_energy", lattice="fcc", n1=8, n2=8, n3=8, S=2, R=2),
        # One trial through the bound Monte Carlo step: configuration up, one
        # trial of the reference stream, configuration down.
        dict(name="mc_step", kind="mc_step", lattice="fcc", n1=8, n2=8, n3=8, S=2, R=2, T=600.0, nbr=False),
        # A bit-exact sequential run of one chain, the energy taken after
        # every sweep (the serial example's loop).
        dict(name="sequential", kind="sequential", lattice="fcc", n1=8, n2=8, n3=8, S=2, R=2, T=600.0, sweeps=4,
             nbr=False),
        # The replica ensemble: one bit-exact chain per rank, many at once.
        dict(name="sequential_replicas", kind="replicas", lattice="fcc", n1=8, n2=8, n3=8, S=2, R=2, T=600.0,
             sweeps=4, chains=128, nbr=False),
        # Energy, pair counts and radial densities of one large quaternary
        # configuration, as a program measures a stored configuration.
        dict(name="measure", kind="measure", lattice="bcc", n1=32, n2=32, n3=32, S=4, R=4),
        # The large quaternary anneal (bcc 32^3, four shells), a few of its
        # temperature steps, radial densities every tenth sweep.
        dict(name="anneal_large", kind="anneal", lattice="bcc", n1=32, n2=32, n3=32, S=4, R=4, T=1100.0,
             dT=-60.0, T_steps=4, sweeps=50, burn=0, rho_every=10),
        # A short run of the small binary lattice, equilibration before the
        # samples, no radial densities.
        dict(name="anneal_small", kind="anneal", lattice="fcc", n1=8, n2=8, n3=8, S=2, R=2, T=600.0, dT=0.0,
             T_steps=1, sweeps=100, burn=20, rho_every=0),
        # Uneven replicas (fcc and bcc, 8 to 24 cells, 2 to 5 species, three
        # shells, 200 to 2000 K), one chain per compute unit.
        dict(name="anneal_batch", kind="anneal_batch", chains=256, lo=8, hi=24, R=3, sweeps=100),
        # One nested-sampling run (quinary fcc 6^3, four shells).
        dict(name="nested", kind="nested", lattice="fcc", n1=6, n2=6, n3=6, S=5, R=4, walkers=128, steps=100,
             iters=100, runs=1),
        # Many nested-sampling runs at once.
        dict(name="nested_batch", kind="nested", lattice="fcc", n1=6, n2=6, n3=6, S=5, R=4, walkers=128, steps=100,
             iters=100, runs=32),
        # One iteration of the Wang-Landau main loop (16 windows of 8 walkers
        # on quaternary bcc 16^3): a sweeps call with window averages, a
        # replica exchange, and the ln g and histograms for the flatness test.
        dict(name="wang_landau", kind="wang_landau", lattice="bcc", n1=16, n2=16, n3=16, S=4, R=2, bins=800,
             windows=16, walkers=8, e_min=-40.0, e_max=10.0, sweeps=1, nbr=False),
        # A mixed stream through the request server, from submission to the
        # last result.
        dict(name="served", kind="served", requests=24, lo=8, hi=20, sweeps=100, walkers=64, iters=50),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi, cubic):
    a = _log_int(rng, lo, hi)
    if cubic:
        return dict(n1=a, n2=a, n3=a)
    return dict(n1=a, n2=_log_int(rng, lo, hi), n3=_log_int(rng, lo, hi))


def draw(rng):
    kind = rng.choice(["pair_energy", "mc_step", "sequential", "replicas", "measure", "anneal", "anneal", "anneal_batch",
                       "nested", "wang_landau", "served"])
    lat = rng.choice(["fcc", "bcc"])
    c = dict(kind=kind, lattice=lat, S=rng.randint(2, 5), R=rng.randint(1, 4))
    if kind == "pair_energy":
        return dict(c, **_box(rng, 4, 16, rng.random() < 0.5))
    if kind in ("mc_step", "sequential", "replicas"):
        c.update(_box(rng, 4, 10, rng.random() < 0.5), T=round(rng.uniform(300.0, 2000.0), 1), nbr=rng.random() < 0.3)
        if kind != "mc_step":
            c.update(sweeps=rng.randint(1, 4))
        if kind == "replicas":
            c.update(chains=_log_int(rng, 16, 128))
        return c
    if kind == "measure":
        return dict(c, **_box(rng, 6, 24 if lat == "fcc" else 32, rng.random() < 0.6))
    if kind == "anneal":
        cubic = rng.random() < 0.75
        c.update(R=rng.randint(2, 4), T=round(rng.uniform(500.0, 2500.0), 1), dT=round(rng.uniform(-60.0, 0.0), 1),
                 T_steps=rng.randint(1, 4), sweeps=_log_int(rng, 10, 50), burn=rng.choice([0, 0, 10]))
        c.update(_box(rng, 8, 24 if cubic else 12, cubic))
        c.update(rho_every=rng.choice([0, 0, 10]) if cubic else 0)
        return c
    if kind == "anneal_batch":
        return dict(kind=kind, chains=_log_int(rng, 16, 256), lo=8, hi=rng.randint(12, 24), R=rng.randint(2, 3),
                    sweeps=_log_int(rng, 20, 100))
    if kind == "nested":
        return dict(c, **_box(rng, 4, 6, rng.random() < 0.6), walkers=_log_int(rng, 32, 128), steps=rng.randint(30, 100),
                    iters=rng.randint(30, 100), runs=_log_int(rng, 1, 16))
    if kind == "wang_landau":
        return dict(c, **_box(rng, 6, 12, True), R=rng.randint(1, 3), S=rng.randint(3, 4),
                    bins=rng.randint(100, 400), windows=rng.randint(1, 4), walkers=rng.randint(2, 8), e_min=-10.0,
                    e_max=10.0, sweeps=rng.randint(1, 3), nbr=rng.random() < 0.3)
    return dict(kind=kind, requests=rng.randint(6, 24), lo=8, hi=rng.randint(10, 20), sweeps=_log_int(rng, 20, 100),
                walkers=_log_int(rng, 32, 64), iters=rng.randint(20, 50))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _sites(lattice, m):
    """Flat Fortran-order indices of a lattice's sites on the doubled grid."""
    x, y, z = np.meshgrid(*[np.arange(k) for k in m], indexing="ij")
    occ = ((x + y + z) % 2 == 0) if lattice == "fcc" else ((x % 2 == y % 2) & (y % 2 == z % 2))
    return np.flatnonzero(occ.ravel(order="F"))


def _random_config(lattice, n, counts, rng):
    m = tuple(2 * k for k in n)
    species = np.repeat(np.arange(1, len(counts) + 1, dtype=np.int8), counts)
    rng.shuffle(species)
    flat = np.zeros(m[0] * m[1] * m[2], dtype=np.int8)
    flat[_sites(lattice, m)] = species
    return flat.reshape(m, order="F")


def _n(c):
    return c["n1"], c["n2"], c["n3"]


def _atoms(lattice, n):
    return (4 if lattice == "fcc" else 2) * n[0] * n[1] * n[2]


def _v(S, R, seed, mev=30.0):
    return _wl.random_v(S, [mev / k for k in range(1, R + 1)], seed)


def _inputs(c, seed):
    """(interactions, configuration) of a one-lattice case, from the seed alone."""
    rng = np.random.Generator(np.random.PCG64(seed))
    n = _n(c)
    v = _v(c["S"], c["R"], seed + 1)
    return v, _random_config(c["lattice"], n, _wl.equal_counts(_atoms(c["lattice"], n), c["S"]), rng), rng


def _two_sites(c, rng):
    m = tuple(2 * k for k in _n(c))
    s = _sites(c["lattice"], m)
    out = []
    for i in rng.choice(len(s), size=2, replace=False):
        x, y, z = np.unravel_index(s[i], m, order="F")
        out.append(np.array([1, x + 1, y + 1, z + 1], dtype=np.int32))
    return out


def _batch_chains(c, seed):
    """A batch of uneven replicas: the boxes and species counts are the case's,
    compositions, interactions, configurations and temperatures the seed's."""
    shape = np.random.Generator(np.random.PCG64([c["chains"], c["lo"], c["hi"]]))
    rng = np.random.Generator(np.random.PCG64(seed))
    out = []
    for k in range(c["chains"]):
        L = int(shape.integers(c["lo"], c["hi"] + 1))
        lat = "fcc" if shape.integers(0, 2) == 0 else "bcc"
        S = int(shape.integers(2, 6))
        N = _atoms(lat, (L, L, L))
        counts = _wl.dirichlet_counts(N, S, rng)
        v = _v(S, c["R"], _wl.derive_seed(seed, k), 25.0)
        cfg = _random_config(lat, (L, L, L), counts, rng)
        p = dict(T=float(rng.uniform(200.0, 2000.0)), n_sweeps=c["sweeps"], seed=_wl.derive_seed(seed + 7, k))
        out.append((lat, (L, L, L), v, cfg, p))
    return out


def _served_requests(c, seed):
    """Six tenths anneals, a quarter nested-sampling runs, the rest short
    Wang-Landau runs; shapes by the case, contents by the seed."""
    shape = np.random.Generator(np.random.PCG64([c["requests"], c["lo"], c["hi"]]))
    rng = np.random.Generator(np.random.PCG64(seed))
    out = []
    for k in range(c["requests"]):
        s = _wl.derive_seed(seed, k)
        u = (k * 7 % 20) / 20.0
        if u < 0.60:
            L = int(shape.integers(c["lo"], c["hi"] + 1))
            lat = "fcc" if shape.integers(0, 2) == 0 else "bcc"
            S = int(shape.integers(2, 6))
            counts = _wl.dirichlet_counts(_atoms(lat, (L, L, L)), S, rng)
            cfg = _random_config(lat, (L, L, L), counts, rng)
            out.append(("anneal", (lat, (L, L, L), _v(S, 3, s, 25.0), cfg),
                        dict(T=float(rng.uniform(200.0, 2000.0)), n_sweeps=c["sweeps"], seed=s, want_config=True)))
        elif u < 0.85:
            out.append(("ns", ("fcc", (6, 6, 6), _v(5, 4, s), s & 0xFFFFFFFF),
                        dict(n_walkers=c["walkers"], n_steps=100, n_iter=c["iters"],
                             species_numbers=_wl.equal_counts(864, 5))))
        else:
            L = int(shape.integers(6, 11))
            out.append(("wl", ("bcc", (L, L, L), _v(4, 2, s)),
                        dict(bins=50, num_windows=1, walkers_per_window=int(shape.integers(4, 9)), bin_overlap=0.1,
                             energy_min=-10.0, energy_max=10.0, mc_sweeps=4, wl_f=1.0, rank_offset=int(s % 1000),
                             species_numbers=_wl.equal_counts(2 * L ** 3, 4))))
    return out


def _walkers_in_windows(c, v, cfg, w, seed):
    """One configuration inside each energy window: a lattice cooled from a
    random start, its configuration kept whenever its energy lies inside a
    window that has none yet (bins in the middle of the window)."""
    found = {}
    lo = [w.bin_edges[int(a) - 1] for a, _ in w.windows]
    hi = [w.bin_edges[int(b)] for _, b in w.windows]
    with _lat.Lattice(c["lattice"], _n(c), v) as L:
        L.set_config(cfg)
        e = L.total_energy()
        for k in range(400):
            for i in range(len(lo)):
                pad = 0.1 * (hi[i] - lo[i])
                if i not in found and lo[i] + pad < e < hi[i] - pad:
                    found[i] = L.get_config()
            if len(found) == len(lo):
                break
            L.metropolis_simulated_annealing(T=6000.0 * 0.982 ** k, n_sweeps=1, seed=seed)
            e = L.total_energy()
        near = sorted(found) or [None]
        for i in range(len(lo)):
            j = min(near, key=lambda q: abs(q - i)) if near[0] is not None else None
            found.setdefault(i, found[j] if j is not None else cfg)
    return [found[i] for i in range(len(lo))]


def prepare(case, seed):
    from brawl_amd.wang_landau import WangLandau
    from brawl_amd.serve import Server
    c, k = case, case["kind"]
    if k == "anneal_batch":
        lats, params = [], []
        for lat, n, v, cfg, p in _batch_chains(c, seed):
            L = _lat.Lattice(lat, n, v)
            L.set_config(cfg)
            lats.append(L)
            params.append(p)
        return dict(case=c, lats=lats, params=params)
    if k == "served":
        return dict(case=c, server=Server(device_bytes=128 << 20, max_launches=8, batch_wait_us=0),
                    requests=_served_requests(c, seed))
    v, cfg, rng = _inputs(c, seed)
    n = _n(c)
    if k == "wang_landau":
        w = WangLandau(c["lattice"], n, v, bins=c["bins"], num_windows=c["windows"], walkers_per_window=c["walkers"],
                       bin_overlap=0.1, energy_min=c["e_min"], energy_max=c["e_max"], mc_sweeps=c["sweeps"],
                       nbr_swap=c["nbr"], rank_offset=seed % 1000)
        for i, start in enumerate(_walkers_in_windows(c, v, cfg, w, seed)):
            for j in range(c["walkers"]):
                w.set_walker(i * c["walkers"] + j, start)
        return dict(case=c, w=w)
    if k in ("replicas", "nested"):
        count = c["chains"] if k == "replicas" else c["runs"]
        lats = []
        for i in range(count):
            L = _lat.Lattice(c["lattice"], n, v)
            L.seed(110179 + 11 * i + seed)
            if k == "replicas":
                counts = _wl.equal_counts(_atoms(c["lattice"], n), c["S"])
                L.set_config(_random_config(c["lattice"], n, counts, rng))
            lats.append(L)
        if k == "replicas":
            return dict(case=c, lats=lats, betas=[_lat.beta_of(c["T"])] * count)
        counts = _wl.equal_counts(_atoms(c["lattice"], n), c["S"])
        return dict(case=c, lats=lats, params=[dict(n_walkers=c["walkers"], n_steps=c["steps"], n_iter=c["iters"],
                                                    species_numbers=counts) for _ in range(count)])
    L = _lat.Lattice(c["lattice"], n, v)
    L.set_config(cfg)
    L.seed(110179 + seed)
    state = dict(case=c, lat=L, cfg=cfg, seed=int(seed))
    if k == "pair_energy":
        state["sites"] = _two_sites(c, rng)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    c = state["case"]
    return globals()["_run_" + c["kind"]](c, state)


def _run_pair_energy(c, st):
    return np.float64(st["lat"].pair_energy(*st["sites"]))


def _run_mc_step(c, st):
    L = st["lat"]
    L.set_config(st["cfg"])
    accept = L.mc_step(_lat.beta_of(c["T"]), nbr_swap=c["nbr"])
    st["cfg"] = L.get_config()
    return accept, st["cfg"]


def _run_sequential(c, st):
    L = st["lat"]
    accepted, energies = L.mc_steps(_lat.beta_of(c["T"]), c["sweeps"] * L.n_atoms, nbr_swap=c["nbr"],
                                    sample_every=L.n_atoms)
    return accepted, energies, L.get_config()


def _run_replicas(c, st):
    lats = st["lats"]
    accepted, energies, _ = _lat.mc_steps_batch(lats, st["betas"], c["sweeps"] * lats[0].n_atoms, nbr_swap=c["nbr"],
                                                sample_every=lats[0].n_atoms)
    return accepted, np.stack(energies), np.stack([L.get_config() for L in lats])


def _run_measure(c, st):
    L = st["lat"]
    return np.float64(L.total_energy()), L.pair_histogram(), L.radial_densities(c["R"] + 1)


def _run_anneal(c, st):
    L = st["lat"]
    r = L.metropolis_simulated_annealing(T=c["T"], delta_T=c["dT"], T_steps=c["T_steps"], n_sweeps=c["sweeps"],
                                         burn_in_sweeps=c["burn"], seed=st["seed"] + 3, asro_every=c["rho_every"])
    return r.energies_of_T, r.C_of_T, r.acceptance_of_T, r.trials, r.accepted, r.rho_of_T, L.get_config()


def _run_anneal_batch(c, st):
    res, _ = _lat.anneal_batch(st["lats"], st["params"])
    return (np.concatenate([r.energies_of_T for r in res]), np.concatenate([r.C_of_T for r in res]),
            np.concatenate([r.acceptance_of_T for r in res]), np.array([r.accepted for r in res]),
            np.concatenate([L.get_config().ravel(order="F") for L in st["lats"]]))


def _run_nested(c, st):
    from brawl_amd.nested_sampling import nested_sampling_batch
    res, _ = nested_sampling_batch(st["lats"], st["params"])
    return np.stack([e for e, _ in res]), np.array([[s.trials, s.accepted] for _, s in res])


def _run_wang_landau(c, st):
    w = st["w"]
    accepted, _ = w.sweeps(1.0)
    partner, exchanged, _ = w.replica_exchange()
    lng, hist = w.lng_hist()
    return accepted, partner, exchanged, lng, hist


def _run_served(c, st):
    srv = st["server"]
    ids = []
    for kind, a, kw in st["requests"]:
        ids.append(getattr(srv, "submit_" + kind)(*a, **kw))
    srv.drain()
    res = [srv.result(i) for i in ids]
    for i in ids:
        del srv.requests[i]
    keys = ("energies_of_T", "C_of_T", "acceptance_of_T", "e_limits", "lng", "hist", "config")
    return {k: np.concatenate([r[k].ravel(order="F") for r in res if k in r]) for k in keys
            if any(k in r for r in res)}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _z(lattice, R):
    return sum(len(_offsets(lattice, d)) for d in SHELLS[lattice][:R])


def work(case):
    c, k = case, case["kind"]
    if k == "anneal_batch":
        atoms = c["chains"] * 3 * ((c["lo"] + c["hi"]) / 2.0) ** 3  # mean of 4 L^3 and 2 L^3
        trials = atoms * c["sweeps"]
        return dict(bytes=2 * atoms, flops=trials * 2 * 0.5 * (_z("fcc", c["R"]) + _z("bcc", c["R"])))
    if k == "served":
        atoms = 0.6 * c["requests"] * 3 * ((c["lo"] + c["hi"]) / 2.0) ** 3
        return dict(bytes=2 * atoms, flops=atoms * c["sweeps"] * 2 * 0.5 * (_z("fcc", 3) + _z("bcc", 3)) +
                    0.25 * c["requests"] * c["iters"] * 100 * 4 * _z("fcc", 4))
    z, n = _z(c["lattice"], c["R"]), _n(c)
    atoms = _atoms(c["lattice"], n)
    v = 8 * c["S"] ** 2 * c["R"]
    if k == "pair_energy":
        return dict(bytes=2 * (z + 1) + v + 8, flops=2 * z)
    if k == "mc_step":
        return dict(bytes=2 * 8 * n[0] * n[1] * n[2] + v, flops=4 * z)
    if k == "measure":
        return dict(bytes=atoms + v, flops=2 * atoms * z)
    # per swap trial of a sequential sampler: both sites' shell sums before
    # and after the swap; of the parallel sampler: both sites' counts
    if k == "sequential":
        return dict(bytes=10 * atoms, flops=c["sweeps"] * atoms * (4 * z + z))
    if k == "replicas":
        return dict(bytes=c["chains"] * 10 * atoms, flops=c["chains"] * c["sweeps"] * atoms * (4 * z + z))
    if k == "anneal":
        return dict(bytes=10 * atoms, flops=c["T_steps"] * (c["sweeps"] + c["burn"]) * atoms * 2 * z)
    if k == "nested":
        return dict(bytes=c["runs"] * (c["walkers"] * atoms + 2 * c["iters"] * atoms),
                    flops=c["runs"] * (c["walkers"] * atoms * z + c["iters"] * c["steps"] * 4 * z))
    walkers = c["windows"] * c["walkers"]
    return dict(bytes=walkers * (2 * atoms + 32 * c["bins"]),
                flops=walkers * atoms * (c["sweeps"] * 4 * z + 2 * z))


# ---------------------------------------------------------------------------
# the same values from numpy alone
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _offsets(lattice, d2):
    """Lattice vectors of squared length d2 on the doubled grid."""
    r = range(-5, 6)
    return [(x, y, z) for x in r for y in r for z in r if x * x + y * y + z * z == d2 and
            ((x + y + z) % 2 == 0 if lattice == "fcc" else x % 2 == y % 2 == z % 2)]


def _site_energy(cfg, v, lattice, R, site):
    m = cfg.shape
    e, a = 0.0, cfg[site] - 1
    for s in range(R):
        for d in _offsets(lattice, SHELLS[lattice][s]):
            e += v[a, cfg[tuple((site[q] + d[q]) % m[q] for q in range(3))] - 1, s]
    return e


def _pair_counts(cfg, lattice, S, R):
    """H(a, b, n): ordered pairs of species (a, b) on shell n."""
    h = np.zeros((S, S, R), dtype=np.int64, order="F")
    at = cfg > 0
    a = cfg[at].astype(np.int64) - 1
    for s in range(R):
        for d in _offsets(lattice, SHELLS[lattice][s]):
            b = np.roll(cfg, (-d[0], -d[1], -d[2]), (0, 1, 2))[at].astype(np.int64) - 1
            h[:, :, s] += np.bincount(a * S + b, minlength=S * S).reshape(S, S)
    return h


def _exact_sequential(c, v, cfg, seed):
    """The sequential chain trial by trial on numpy's MT19937; None where a
    trial's energy change is zero but for rounding, so that the order of the
    additions decides whether a random number is drawn (binary lattices)."""
    n, R, lattice = _n(c), c["R"], c["lattice"]
    m = cfg.shape
    atoms = _atoms(lattice, n)
    trials = c["sweeps"] * atoms
    shell_of, off = [], []
    for s in range(R):
        for d in _offsets(lattice, SHELLS[lattice][s]):
            shell_of.append(s)
            off.append(d)
    shell_of, off = np.array(shell_of), np.array(off)
    near = [(1, 1, 1), (1, 1, -1), (1, -1, 1), (1, -1, -1), (-1, 1, 1), (-1, 1, -1), (-1, -1, 1), (-1, -1, -1)] \
        if lattice == "bcc" else \
        [(0, 1, 1), (0, 1, -1), (0, -1, 1), (0, -1, -1), (1, 1, 0), (1, -1, 0), (1, 0, 1), (1, 0, -1), (-1, 1, 0),
         (-1, -1, 0), (-1, 0, 1), (-1, 0, -1)]
    gen = np.random.MT19937()
    gen._legacy_seeding(110179 + seed)
    u = gen.random_raw(7 * trials).astype(np.float64) / 4294967296.0
    at = 0
    mm = np.array(m)

    def site():
        nonlocal at
        k = int(2 * u[at] * n[2])
        if lattice == "bcc":
            x, y = 2 * int(u[at + 1] * n[0]) + (k & 1), 2 * int(u[at + 2] * n[1]) + (k & 1)
        else:
            x = int(2 * u[at + 1] * n[0])
            y = 2 * int(u[at + 2] * n[1]) + ((x + k) & 1)
        at += 3
        return x, y, k

    def energy(s, a):
        p = (off + np.array(s)) % mm
        return float(v[a - 1, cfg[p[:, 0], p[:, 1], p[:, 2]] - 1, shell_of].sum())

    beta = _lat.beta_of(c["T"])
    cfg = cfg.copy(order="F")
    energies = []
    for t in range(1, trials + 1):
        s1 = site()
        if c["nbr"]:
            d = near[int(len(near) * u[at])]
            at += 1
            s2 = tuple((s1[q] + d[q]) % m[q] for q in range(3))
        else:
            s2 = site()
        a, b = cfg[s1], cfg[s2]
        if a != b:
            before = energy(s1, a) + energy(s2, b)
            cfg[s1], cfg[s2] = b, a
            de = energy(s1, b) + energy(s2, a) - before
            if abs(de) < 1e-14:
                return None
            if de >= 0.0:
                r = u[at]
                at += 1
                if not r < math.exp(-beta * de):
                    cfg[s1], cfg[s2] = a, b
        if t % atoms == 0:
            energies.append(0.5 * float((_pair_counts(cfg, lattice, c["S"], R) * v).sum()))
    return np.array(energies)


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "pair_energy":
        v, cfg, rng = _inputs(c, seed)
        return np.float64(sum(_site_energy(cfg, v, c["lattice"], c["R"], tuple(int(q) - 1 for q in s[1:]))
                              for s in _two_sites(c, rng)))
    if k == "measure":
        v, cfg, _ = _inputs(c, seed)
        S, R = c["S"], c["R"]
        h = _pair_counts(cfg, c["lattice"], S, R)
        counts = np.bincount(cfg[cfg > 0].astype(np.int64) - 1, minlength=S).astype(np.float64)
        rho = np.zeros((S, S, R + 1), order="F")
        rho[:, :, 0] = np.eye(S)
        rho[:, :, 1:] = h / counts[:, None, None]
        return np.float64(0.5 * (h * v).sum()), h, rho
    if k == "sequential" and c["sweeps"] * _atoms(c["lattice"], _n(c)) <= 60000:
        v, cfg, _ = _inputs(c, seed)
        energies = _exact_sequential(c, v, cfg, seed)
        return None if energies is None else (None, energies, None)
    # The other samplers' outputs are averages over a random trajectory that
    # the library's own streams and summation orders define.
    return None
