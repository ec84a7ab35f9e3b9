"""A chain that could be divided over workgroups (bwl_metro_split.hip) while
another process holds most of the device."""
import subprocess
import sys
import time

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from brawl_amd import _lib
    L = _lib.load()
    if _lib.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return L


def _lattice():
    from brawl_amd import Lattice, workloads
    n, S = (32, 32, 32), 4
    L = Lattice(2, n, workloads.random_v(S, [25.0 / k for k in range(1, 5)], 7))
    L.set_config(workloads.random_config(2, n, workloads.equal_counts(L.n_atoms, S), np.random.default_rng(7)))
    return L


OTHER = """
import sys
sys.path.insert(0, {root!r})
import numpy as np
from brawl_amd import Lattice, anneal_batch, workloads
v = workloads.random_v(2, [25.0, 12.5], 3)
cfg = workloads.random_config(1, (16, 16, 16), workloads.equal_counts(16384, 2), np.random.default_rng(1))
chains = []
for k in range(200):
    L = Lattice(1, (16, 16, 16), v)
    L.set_config(cfg)
    chains.append(L)
ps = [dict(T=900.0, n_sweeps=40, seed=k) for k in range(200)]
anneal_batch(chains, ps)
print("go", flush=True)
anneal_batch(chains, [dict(p, n_sweeps=30000) for p in ps])
print("end", flush=True)
"""


def test_another_process_holds_the_cus(lib):
    """200 CUs are another process's for seconds: the parts of a chain do not
    all arrive, and the call takes little longer than undivided (a wait of 1 s
    for the parts before)."""
    with _lattice() as L:
        p = dict(T=900.0, n_sweeps=40, seed=1)
        L.metropolis_simulated_annealing(**p)
        child = subprocess.Popen([sys.executable, "-c", OTHER.format(root=ROOT)], stdout=subprocess.PIPE, text=True)
        try:
            assert child.stdout.readline().strip() == "go"
            time.sleep(0.3)
            t = time.perf_counter()
            L.metropolis_simulated_annealing(**p)
            took = time.perf_counter() - t
            alone_in_time = child.poll() is None
            assert child.stdout.readline().strip() == "end" and child.wait(60) == 0
        finally:
            if child.poll() is None:
                child.terminate()
        print(f"{took * 1e3:.1f} ms")
        assert alone_in_time
        assert took < 0.5
