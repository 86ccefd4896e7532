"""FP32 M2L with one wave per work item (m2l_wave32.hip) against FP64 plans.

Three chains of FP32 products with up to 2 (p + 1) terms each (random signs: about 3 sqrt(30) of
2^-24, 1e-6 of the far field), expansions rounded to FP32 once; the near field of a mixed plan adds
a few 2^-24: 2e-6 of the l2 norm in all."""
import numpy as np
import pytest

from oracle import direct as D

pytestmark = pytest.mark.gpu
TOL = 2e-6


@pytest.fixture(scope="module")
def hf():
    import hfmm0_amd
    return hfmm0_amd


def _points(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "cube":
        x = rng.uniform(size=(n, 3))
    else:   # a sphere and two clusters: uneven levels
        v = rng.normal(size=(n // 2, 3))
        c = np.array([[0.2, 0.3, 0.7], [0.81, 0.2, 0.4]])
        x = np.vstack([0.5 + 0.45 * v / np.linalg.norm(v, axis=1, keepdims=True),
                       c[rng.integers(0, 2, n - n // 2)] + rng.normal(scale=0.01, size=(n - n // 2, 3))])
    return x, rng.normal(size=n) + 1j * rng.normal(size=n)


@pytest.mark.parametrize("p", list(range(2, 16)))
def test_degrees(hf, p):
    """Every degree of the kernel and the first one past it (15), on uneven levels."""
    print(f"case: wave32 p={p}", flush=True)
    x, q = _points("surface", 5000, p)
    ref = hf.evaluate(hf.setup(x, 6.0, p=p, N_max=24), q)
    assert D.relative_error(hf.evaluate(hf.setup(x, 6.0, p=p, N_max=24, precision="mixed"), q), ref) < TOL


@pytest.mark.parametrize("levels,k", [([6, 6, 9, 4, 3], 4.0), ([14, 14, 5, 13, 8], -11.0), ([3, 3, 3, 14, 2], 0.0)])
def test_level_degrees(hf, levels, k):
    """Degrees that differ between levels, then lowered for an evaluate and raised again."""
    print(f"case: wave32 degrees {levels} k={k}", flush=True)
    x, q = _points("cube", 12000, 3)
    st = hf.setup(x, k, p=max(levels), N_max=16, p_level=levels, precision="mixed")
    ref = hf.setup(x, k, p=max(levels), N_max=16, p_level=levels)
    full = hf.evaluate(ref, q)
    assert D.relative_error(hf.evaluate(st, q), full) < TOL
    low = [max(2, v - 2) for v in levels[:st.depth]]
    for s in (st, ref):
        s.set_degrees(low)
    assert D.relative_error(hf.evaluate(st, q), hf.evaluate(ref, q)) < TOL
    for s in (st, ref):
        s.set_degrees([0] * s.depth)
    assert D.relative_error(hf.evaluate(st, q), full) < TOL


def test_many_blocks(hf):
    """A level with more blocks than items (whole blocks), and levels split over items."""
    print("case: wave32, 150000 points in leaves of 8", flush=True)
    x, q = _points("cube", 150000, 5)
    st = hf.setup(x, 9.0, p=4, N_max=8, precision="mixed", tree_device=True)
    assert D.relative_error(hf.evaluate(st, q), hf.evaluate(hf.setup(x, 9.0, p=4, N_max=8, tree_device=True), q)) < TOL
