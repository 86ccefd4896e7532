"""Which levels the one-wave-per-item kernels take, and their results there against other kernels:
M2M and L2L with unequal and lowered degrees (FP64), the last degree of each kernel and the first
past it, and near-field chunks of every size up to the largest."""
import numpy as np
import pytest

from oracle import direct as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hf():
    import hfmm0_amd
    return hfmm0_amd


def _cube(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(size=(n, 3)), rng.normal(size=n) + 1j * rng.normal(size=n)


def test_tree_levels_of_unequal_degrees(hf):
    """600000 points, depth 6: M2M into and L2L out of levels 4 and 5 on the wave kernel, with the
    source's degree above and below the target's, then lowered; the generic kernel is the reference
    (the same products in FP64: 1e-13)."""
    x, q = _cube(600000, 3)
    for levels in ([4, 4, 4, 7, 3, 6], [5, 5, 6, 3, 6, 3]):
        print(f"case: M2M and L2L degrees {levels}", flush=True)
        kw = dict(p=7, N_max=1, max_depth=6, tree_device=True, p_level=levels)
        s, g = hf.setup(x, 5.0, **kw), hf.setup(x, 5.0, m2l_kernel="generic", **kw)
        w = s.wave_levels()
        assert w["m2m"] == [4, 5] and w["l2l"] == [4, 5] and w["m2l"] == [2, 3, 4, 5, 6], w
        assert g.wave_levels() == {"m2l": [], "m2m": [], "l2l": []}
        assert D.relative_error(hf.evaluate(s, q), hf.evaluate(g, q)) < 1e-13
        low = [max(2, v - 1 - i % 2) for i, v in enumerate(levels)]
        for st in (s, g):
            st.set_degrees(low)
        assert D.relative_error(hf.evaluate(s, q), hf.evaluate(g, q)) < 1e-13
        s.close()
        g.close()


@pytest.mark.parametrize("precision,last", [("fp64", 14), ("mixed", 15)])
def test_last_degree_and_the_first_past_it(hf, precision, last):
    """Past the wave kernel the block kernel takes the level.  FP64: 1e-13 of the generic kernel.
    Mixed: 2e-6, the bound of the FP32 M2L's own test."""
    x, q = _cube(6000, 7)
    for p in (2, last, last + 1):
        print(f"case: {precision} p={p}", flush=True)
        st = hf.setup(x, 4.0, p=p, N_max=16, precision=precision)
        assert st.wave_levels()["m2l"] == (list(range(2, st.depth + 1)) if p <= last else [])
        assert st.m2l_fp32_levels == (list(range(2, st.depth + 1)) if precision == "mixed" else [])
        ref = hf.evaluate(hf.setup(x, 4.0, p=p, N_max=16, m2l_kernel="generic"), q)
        assert D.relative_error(hf.evaluate(st, q), ref) < (1e-13 if precision == "fp64" else 2e-6)


@pytest.mark.parametrize("n", [36000, 70001, 140000])
def test_large_near_field_chunks(hf, n):
    """Eight leaves, every pair near: chunks of 32, 64 and 128 targets (a thousandth of the launch's
    pairs is that many targets' here), against the oracle at 64 targets.  Sums of n terms: the direct
    sum's 1e-13, the field's 1e-12, mixed 2e-6."""
    x, q = _cube(n, 11)
    idx = np.sort(np.random.default_rng(1).choice(n, 64, replace=False))
    ref, eref = D.direct_c(x, q, 6.0, idx), D.direct_field_c(x, q, 6.0, idx)
    for precision, tol in (("fp64", 1e-13), ("mixed", 2e-6)):
        print(f"case: near field alone, {n} points, {precision}", flush=True)
        st = hf.setup(x, 6.0, p=4, N_max=n, max_depth=1, precision=precision)
        assert st.depth == 1
        assert D.relative_error(hf.evaluate(st, q)[idx], ref) < tol
        phi, e = hf.evaluate_field(st, q)
        assert D.relative_error(phi[idx], ref) < tol
        assert D.relative_error(e[idx], eref) < max(tol, 1e-12)
        st.close()


def test_cluster_alone(hf):
    """A cluster of 600 among 2000 points, eight leaves: one leaf with most of the pairs, split into
    the smallest chunks, beside leaves left whole."""
    print("case: near field of a cluster", flush=True)
    rng = np.random.default_rng(2)
    x = np.vstack([rng.uniform(size=(2000, 3)), 0.3 + 1e-3 * rng.uniform(size=(600, 3))])
    q = rng.normal(size=len(x)) + 1j * rng.normal(size=len(x))
    st = hf.setup(x, 3.0, p=4, N_max=2600, max_depth=1)
    assert D.relative_error(hf.evaluate(st, q), D.direct_c(x, q, 3.0)) < 1e-13


@pytest.mark.parametrize("n,p,precision,wave", [(26, 2, "fp64", False), (26, 9, "fp64", False), (100, 9, "fp64", True),
                                                (52, 13, "fp64", True), (52, 14, "fp64", False), (100, 14, "fp64", True),
                                                (8, 2, "mixed", True), (8, 10, "mixed", True), (8, 11, "mixed", False),
                                                (26, 14, "mixed", False), (52, 14, "mixed", True), (52, 15, "mixed", True),
                                                (40, 15, "mixed", False)])
def test_small_levels(hf, n, p, precision, wave):
    """One M2L level of 34 pairs (8 points) to 1886 (100 points): few pairs stay on the block kernel,
    whose time they are (a whole evaluate of 26 points at p = 9 took 62 us on the wave kernel, 53 on the
    block kernel).  In a batch the FP64 level takes the wave kernel at any size."""
    from hfmm0_amd.batch import Batch
    print(f"case: one small M2L level, {n} points, p={p}, {precision}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(size=(n, 3))
    x[0], x[1] = 0.001, 0.999
    q = rng.normal(size=n) + 1j * rng.normal(size=n)
    kw = dict(p=p, N_max=1, max_depth=2, precision=precision)
    st = hf.setup(x, 6.0, **kw)
    assert st.depth == 2 and st.wave_levels()["m2l"] == ([2] if wave else [])
    kw["precision"] = "fp64"
    ref = hf.evaluate(hf.setup(x, 6.0, m2l_kernel="generic", **kw), q)
    tol = 1e-13 if precision == "fp64" else 2e-6
    phi = hf.evaluate(st, q)
    assert D.relative_error(phi, ref) < tol
    kw["precision"] = precision
    kw.pop("max_depth")
    B = Batch([x, x], [6.0, 6.0], max_depth=2, **kw)
    assert B.plan(0).wave_levels()["m2l"] == ([2] if wave or precision == "fp64" else [])
    for v in B.evaluate([q, q]):
        assert D.relative_error(v, ref) < tol
    B.close()


@pytest.mark.parametrize("p,m2m,l2l", [(10, True, True), (11, False, True), (13, False, True), (14, False, False)])
def test_tree_levels_by_degree(hf, p, m2m, l2l):
    """M2M runs on the wave kernel up to p = 10 and L2L up to 13, where the block kernel is slower; a
    level at a higher degree on either side counts as that degree.  Results against the generic kernel."""
    print(f"case: tree levels at p={p}", flush=True)
    x, q = _cube(250000, p)
    levels = [4, 4, 4, p, 4, 4]            # levels 3 -> 4 and 4 -> 5 with degree p on one side
    kw = dict(p=p, N_max=1, max_depth=6, tree_device=True, p_level=levels)
    s = hf.setup(x, 5.0, **kw)
    w = s.wave_levels()
    assert (4 in w["m2m"]) == m2m and (4 in w["l2l"]) == l2l, w
    assert 5 in w["m2m"] and 5 in w["l2l"], w
    assert D.relative_error(hf.evaluate(s, q), hf.evaluate(hf.setup(x, 5.0, m2l_kernel="generic", **kw), q)) < 1e-13
