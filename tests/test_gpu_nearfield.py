"""Near field by work items (nearfield.hip) where its chunks, batches and item splits have edges.

Points few enough for one leaf are a pure near field.  Tolerances: FP64 sums n terms of relative
error a few 2^-52: 1e-13 (field, whose terms cancel more: 1e-12).  Mixed: each FP32 weight and
product carries a few 2^-24 relative to its term, 64-term FP32 sums as many again: 2e-6 of the l2
norm (charges random, terms add in quadrature)."""
import numpy as np
import pytest

from oracle import direct as D

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 130, 191, 257, 300]


@pytest.fixture(scope="module")
def hf():
    import hfmm0_amd
    return hfmm0_amd


def _cloud(n, seed=0):
    rng = np.random.default_rng(seed + n)
    return rng.uniform(size=(n, 3)), rng.normal(size=n) + 1j * rng.normal(size=n)


def _direct(x, q, k):
    d = np.linalg.norm(x[:, None] - x[None], axis=2)
    np.fill_diagonal(d, np.inf)
    return (np.where(np.isinf(d), 0, np.exp(1j * k * np.where(np.isinf(d), 0, d)) / d)) @ q


def _direct_field(x, q, k):
    r = x[:, None] - x[None]
    d = np.linalg.norm(r, axis=2)
    np.fill_diagonal(d, 1.0)
    w = (1 - 1j * k * d) * np.exp(1j * k * d) / d ** 3
    np.fill_diagonal(w, 0)
    return np.einsum("ijc,ij,j->ic", r, w, q)


@pytest.mark.parametrize("precision,k,tile", [("fp64", 9.0, 0), ("mixed", 0.0, 0), ("mixed", 5.0, 0), ("mixed", -5.0, 1),
                                              ("mixed", 5.0, 4), ("mixed", 60.0, 0), ("mixed", 60.0, 1), ("mixed", 0.0, 4)])
def test_chunks(hf, precision, k, tile):
    tol = 1e-13 if precision == "fp64" else 2e-6
    for n in SIZES:
        print(f"case: one leaf n={n} {precision} k={k} tile={tile}", flush=True)
        x, q = _cloud(n)
        st = hf.setup(x, k, p=4, N_max=512, precision=precision, p2p_tile=tile)
        phi = hf.evaluate(st, q)
        ref = _direct(x, q, k)
        assert np.linalg.norm(phi - ref) <= tol * max(np.linalg.norm(ref), np.finfo(float).tiny)


@pytest.mark.parametrize("precision,k", [("fp64", 9.0), ("mixed", 5.0), ("mixed", 60.0)])
def test_field_chunks(hf, precision, k):
    tol = 1e-12 if precision == "fp64" else 2e-6
    for n in SIZES:
        print(f"case: one leaf with field n={n} {precision} k={k}", flush=True)
        x, q = _cloud(n)
        q = q.real.copy()
        phi, e = hf.evaluate_field(hf.setup(x, k, p=4, N_max=512, precision=precision), q)
        for got, ref in ((phi, _direct(x, q, k)), (e, _direct_field(x, q, k))):
            assert np.linalg.norm(got - ref) <= tol * max(np.linalg.norm(ref), np.finfo(float).tiny)


@pytest.mark.parametrize("n_max", [1, 40, 200])
def test_split_leaves(hf, n_max):
    """A spread cloud and a tight cluster: leaves with many small ranges (several in a batch of 64)
    and leaves whose chunks are halved.  Degree 20 at k = 2 leaves the far field's error below 1e-9
    (each degree gains a factor 2 or more from 1)."""
    print(f"case: cluster, leaf {n_max}", flush=True)
    rng = np.random.default_rng(n_max)
    n = 2500
    x = np.vstack([rng.uniform(size=(n - 200, 3)), 0.3 + 1e-3 * rng.uniform(size=(200, 3))])
    x = np.vstack([x, [0.05, 0.05, 0.05] + 0.02 * rng.uniform(size=(600, 3))])
    q = rng.normal(size=len(x)) + 1j * rng.normal(size=len(x))
    phi = hf.evaluate(hf.setup(x, 2.0, p=20, N_max=n_max), q)
    assert D.relative_error(phi, _direct(x, q, 2.0)) < 1e-6
