"""GPU test of L2P by runs of levels: leaves of levels with different degrees, evaluated in launches
of their own, give what one launch over all leaves gives (a plan whose tables have one degree at
every level and is set to the same degrees)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degrees", [(8, 8, 8, 8, 8, 7, 6), (6, 6, 6, 6, 6, 7, 8), (8, 7, 6, 7, 8, 7, 6)])
@pytest.mark.parametrize("n,leaf", [(150_001, 8), (20_000, 16), (300, 16)])
def test_runs_of_levels_equal_one_launch(n, leaf, degrees):
    import hfmm0_amd as hf
    print(f"case: l2p runs n={n} leaf={leaf} degrees={degrees}", flush=True)
    rng = np.random.default_rng(5)
    centres = rng.uniform(0.2, 0.8, (4, 3))
    x = np.vstack([rng.uniform(0.0, 1.0, (n // 2, 3)),
                   centres[rng.integers(0, 4, n - n // 2)] + rng.normal(scale=0.06, size=(n - n // 2, 3))])
    q = rng.normal(size=n) + 1j * rng.normal(size=n)
    runs = hf.setup(x, 3.0, p=8, N_max=leaf, p_level=list(degrees) + [degrees[-1]] * 8, max_depth=8)
    one = hf.setup(x, 3.0, p=8, N_max=leaf, max_depth=8)
    one.set_degrees((list(degrees) + [degrees[-1]] * 8)[:one.depth])
    a, b = hf.evaluate(runs, q), hf.evaluate(one, q)
    runs.close()
    one.close()
    # the same sums in FP64; tables of another size may round in another order: a few hundred
    # roundings of 1.1e-16 per value
    assert np.linalg.norm(a - b) <= 1e-13 * np.linalg.norm(b)
