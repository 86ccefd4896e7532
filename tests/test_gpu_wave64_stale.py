"""FP64 wave translations read the coefficients of the effective degrees and nothing else: what an
earlier call left above them, or in the box that follows in memory, does not reach the result.

A call with a NaN charge leaves NaN in every coefficient that it writes; the next call has finite
charges and is compared with a plan of its own (the same sums in FP64, tables of another size may
round in another order: 1e-13)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hf():
    import hfmm0_amd
    return hfmm0_amd


def _problem(n, seed):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=(n // 2, 3))
    x = np.vstack([0.5 + 0.45 * v / np.linalg.norm(v, axis=1, keepdims=True), rng.uniform(size=(n - n // 2, 3))])
    return x, rng.normal(size=n) + 1j * rng.normal(size=n)


def _rel(a, b):
    assert np.isfinite(b).all()
    assert np.isfinite(a).all(), f"{np.count_nonzero(~np.isfinite(a))} values are not finite"
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("p", range(2, 14))
def test_lowered_after_bad_charges(hf, p, bad):
    print(f"case: wave64 tables of degree {p + 1}, lowered to {p} after a charge {bad}", flush=True)
    x, q = _problem(3000, p)
    st = hf.setup(x, 5.0, p=p + 1, N_max=24)
    poison = q.copy()
    poison[1234] = bad
    assert not np.isfinite(hf.evaluate(st, poison)).all()
    st.set_degrees([p] * st.depth)
    assert _rel(hf.evaluate(st, q), hf.evaluate(hf.setup(x, 5.0, p=p, N_max=24), q)) < 1e-13


@pytest.mark.parametrize("p", range(2, 14))
def test_lowered_before_the_first_call(hf, p):
    """Coefficients above the effective degree that no call has written."""
    print(f"case: wave64 tables of degree {p + 1}, lowered to {p} at once", flush=True)
    x, q = _problem(3000, p)
    st = hf.setup(x, 5.0, p=p + 1, N_max=24)
    st.set_degrees([p] * st.depth)
    assert _rel(hf.evaluate(st, q), hf.evaluate(hf.setup(x, 5.0, p=p, N_max=24), q)) < 1e-13


@pytest.mark.parametrize("p", [2, 4, 5])
def test_call_after_bad_charges(hf, p):
    """M2M and L2L on the wave kernel at two levels each (600000 points, depth 6): the last box of a
    level is followed by the next level's first, which still holds the previous call's values."""
    print(f"case: wave64 tree translations p={p}, a call after a NaN charge", flush=True)
    rng = np.random.default_rng(p)
    x = rng.uniform(size=(600000, 3))
    q = rng.normal(size=len(x))
    st = hf.setup(x, 3.0, p=p, N_max=1, max_depth=6, tree_device=True)
    assert st.depth == 6
    w = st.wave_levels()
    assert w["m2m"] == [4, 5] and w["l2l"] == [4, 5], w
    first = hf.evaluate(st, q)
    q2 = q.copy()
    q2[::7] = np.nan
    assert not np.isfinite(hf.evaluate(st, q2)).any()
    assert _rel(hf.evaluate(st, q), first) < 1e-13


def test_batch_after_bad_charges(hf):
    from hfmm0_amd.batch import Batch
    print("case: wave64 batch, lowered after a NaN charge", flush=True)
    probs = [_problem(n, n) for n in (900, 2500, 4100)]
    B = Batch([x for x, _ in probs], [5.0] * len(probs), p=9, N_max=32)
    B.evaluate([np.where(np.arange(len(q)) == 5, np.nan, q) for _, q in probs])
    for i in range(len(probs)):
        B.plan(i).set_degrees([8] * B.plan(i).depth)
    for (x, q), phi in zip(probs, B.evaluate([q for _, q in probs])):
        assert _rel(phi, hf.evaluate(hf.setup(x, 5.0, p=8, N_max=32), q)) < 1e-13
