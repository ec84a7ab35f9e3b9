"""A walker's set-up that takes more draws than the device makes for one: the
concentrations add up to little, so most draws name no species."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,conc", [((24, 24, 24), [2e-4, 2e-4]), ((10, 10, 10), [4e-4, 6e-4]), ((10, 10, 10), [0.2, 0.3])])
def test_concentrations_that_add_up_to_little(oracle, n, conc):
    """69 million draws a walker on the mean (refused when drawn on the
    device), 2 million, and 4000."""
    from brawl_amd import Lattice, nested_sampling, workloads
    print("case", n, conc, flush=True)
    v = workloads.random_v(2, [30.0], 5)
    p = dict(n_walkers=2, n_steps=2, n_iter=1, concentrations=np.array(conc))
    ref = oracle.OracleLattice(2, n, v)
    gen = oracle.Generator(4357)
    lim_ref = ref.nested_sampling(gen, **p)
    with Lattice(2, n, v) as L:
        L.seed(4357)
        lim, _ = nested_sampling.nested_sampling(L, **p)
        state = L.genrand_state()
    assert np.array_equal(lim, lim_ref)
    mt, mti = gen.state_arrays()
    assert state[1] == mti and np.array_equal(state[0], mt)
