"""FP64 translations with one wave per work item (m2l_wave64.hip) against the generic kernel.

Both sum the same products in FP64 in different orders, so the results agree to FP64 rounding:
the bound is 1e-13 relative, the one of the block kernel's own comparison."""
import numpy as np
import pytest

from oracle import direct as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hf():
    import hfmm0_amd
    return hfmm0_amd


def _points(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "cube":
        x = rng.uniform(size=(n, 3))
    else:   # a sphere and two clusters: W and X lists, levels with few and uneven targets
        v = rng.normal(size=(n // 2, 3))
        c = np.array([[0.2, 0.3, 0.7], [0.81, 0.2, 0.4]])
        x = np.vstack([0.5 + 0.45 * v / np.linalg.norm(v, axis=1, keepdims=True),
                       c[rng.integers(0, 2, n - n // 2)] + rng.normal(scale=0.01, size=(n - n // 2, 3))])
    return x, rng.normal(size=n) + 1j * rng.normal(size=n)


def _pair(hf, x, q, k, **kw):
    out = []
    for m in ("auto", "generic"):
        st = hf.setup(x, k, m2l_kernel=m, **kw)
        out.append((st, hf.evaluate(st, q)))
    return out


@pytest.mark.parametrize("p", list(range(2, 16)))
def test_degrees(hf, p):
    """Every degree of the kernel and the first one past it (15), on uneven levels."""
    print(f"case: wave64 p={p}", flush=True)
    x, q = _points("surface", 5000, p)
    (_, a), (_, b) = _pair(hf, x, q, 6.0, p=p, N_max=24)
    assert D.relative_error(a, b) < 1e-13


@pytest.mark.parametrize("levels,k", [([6, 6, 9, 4, 3], 4.0), ([14, 14, 5, 13, 8], -11.0), ([3, 3, 3, 15, 2], 0.0)])
def test_level_degrees(hf, levels, k):
    """Source and target degrees that differ between levels, then lowered for an evaluate."""
    print(f"case: wave64 degrees {levels} k={k}", flush=True)
    x, q = _points("cube", 12000, 3)
    (s, a), (g, b) = _pair(hf, x, q, k, p=max(levels), N_max=16, p_level=levels)
    assert D.relative_error(a, b) < 1e-13
    low = [max(2, v - 2) for v in levels[:s.depth]]
    for st in (s, g):
        st.set_degrees(low)
    assert D.relative_error(hf.evaluate(s, q), hf.evaluate(g, q)) < 1e-13
    for st in (s, g):
        st.set_degrees([0] * st.depth)
    assert D.relative_error(hf.evaluate(s, q), b) < 1e-13


def test_tree_translations(hf):
    """A finest level of 32768 boxes: M2M and L2L take the kernel too (2048 groups)."""
    print("case: wave64 M2M and L2L, depth 5", flush=True)
    x, q = _points("cube", 120000, 5)
    (s, a), (_, b) = _pair(hf, x, q, 9.0, p=4, N_max=8, tree_device=True)
    assert s.depth == 5
    assert D.relative_error(a, b) < 1e-13


def test_batch(hf):
    """Problems of different degrees and sizes in one batch, against each alone, twice (replay)."""
    from hfmm0_amd.batch import Batch
    print("case: wave64 batch", flush=True)
    probs = [_points(kind, n, n) for kind, n in (("cube", 900), ("surface", 4100), ("cube", 9001), ("surface", 2500))]
    ps = [[5] * 8, [8] * 8, [10] * 8, [14, 14, 9, 7, 6, 5, 5, 5]]
    ks = [3.0, 7.0, 0.0, 12.0]
    B = Batch([x for x, _ in probs], ks, p=14, N_max=32, p_level=ps)
    for rep in range(2):
        out = B.evaluate([q * (1 + rep) for _, q in probs])
        for (x, q), k, pl, phi in zip(probs, ks, ps, out):
            alone = hf.evaluate(hf.setup(x, k, p=14, N_max=32, p_level=pl), q * (1 + rep))
            assert D.relative_error(phi, alone) < 1e-13


def test_batch_plan_alone(hf):
    """A problem of a batch evaluated by itself runs its own work items, before and after the batch."""
    from hfmm0_amd.batch import Batch
    print("case: wave64 batch, its plans alone", flush=True)
    probs = [_points("cube", 3000, 1), _points("surface", 4100, 2)]
    B = Batch([x for x, _ in probs], [5.0, 7.0], p=8, N_max=32)
    for rep in range(2):
        for i, (x, q) in enumerate(probs):
            alone = hf.evaluate(hf.setup(x, [5.0, 7.0][i], p=8, N_max=32), q)
            assert D.relative_error(hf.evaluate(B.plan(i), q), alone) < 1e-13
        B.evaluate([q for _, q in probs])
