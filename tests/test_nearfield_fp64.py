"""FP64 near-field weight (hfmm0_amd/csrc/p2p_math.h) built for the host, and the GPU kernels
that use it, against plain FP64 and extended-precision references.

Host bounds, from the roundings: 1/r carries the cubic correction's last rounding (2^-53) and
that of its product terms (below 2 ulp in all), r one rounding of its correction (1 ulp); sin and
cos of pi y the Remez error (1.3e-16) and about two roundings of values up to pi / 2 (4e-16 each).
A weight's phase is r k/pi reduced with k/pi in two terms: the error of r (2^-52 relative) times
k r, plus the polynomials' 1e-15.
"""
import ctypes
import os
import subprocess
import tempfile

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EPS = 2.0 ** -52


@pytest.fixture(scope="module")
def nf():
    so = os.path.join(tempfile.mkdtemp(prefix="nf64_"), "libnf64.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-march=x86-64-v3", "-ffp-contract=off", "-fPIC", "-shared",
                    os.path.join(HERE, "native", "nearfield64_host.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def test_rsqrt64(nf):
    r2 = np.concatenate([np.geomspace(2.0 ** -1022, 1e300, 200001), np.linspace(0.5, 4.0, 100001)])
    rinv, r = np.empty_like(r2), np.empty_like(r2)
    nf.nf64_rsqrt(_p(r2), ctypes.c_int(len(r2)), _p(rinv), _p(r))
    ref = np.sqrt(r2.astype(np.longdouble))
    assert np.max(np.abs(r / ref - 1)) <= 1.0 * EPS
    assert np.max(np.abs(rinv * ref - 1)) <= 2.0 * EPS


def test_sincospi_half64(nf):
    y = np.linspace(-0.5, 0.5, 400001)
    s, c = np.empty_like(y), np.empty_like(y)
    nf.nf64_sincospi(_p(y), ctypes.c_int(len(y)), _p(s), _p(c))
    pi = np.longdouble("3.14159265358979323846264338327950288")
    yl = y.astype(np.longdouble)
    assert np.max(np.abs(s - np.sin(pi * yl))) < 6e-16
    assert np.max(np.abs(c - np.cos(pi * yl))) < 6e-16
    sm, cm, ym = np.empty_like(y), np.empty_like(y), -y
    nf.nf64_sincospi(_p(ym), ctypes.c_int(len(y)), _p(sm), _p(cm))
    assert np.array_equal(sm, -s) and np.array_equal(cm, c)
    assert s[len(y) // 2] == 0.0 and c[len(y) // 2] == 1.0


@pytest.mark.parametrize("k", [0.0, 1e-3, 3.0, 40.0, 1234.5])
def test_pair_weight64(nf, k):
    r = np.concatenate([np.geomspace(1e-9, 1.0, 100001), np.linspace(1.0, 20.0, 100001)])
    r2 = r * r
    wr, wi = np.empty_like(r), np.empty_like(r)
    nf.nf64_weight(_p(r2), ctypes.c_int(len(r)), ctypes.c_double(0.0), ctypes.c_double(k), _p(wr), _p(wi))
    rl = np.sqrt(r2.astype(np.longdouble))
    ph = np.longdouble(k) * rl
    err = np.hypot((wr * rl - np.cos(ph)).astype(float), (wi * rl - np.sin(ph)).astype(float))
    assert np.all(err <= 4 * EPS + 1e-15 + (k * r) * 2 * EPS), float(np.max(err))
    if k == 0.0:
        assert np.all(wi == 0.0)


def test_pair_weight64_edges(nf):
    # zero at and below the floor; finite at r = 0, at the smallest normal r^2 and far beyond
    # the reduction's range; NaN where r^2 overflowed, as an FP64 e^{ikr}/r gives
    r2 = np.array([0.0, 5e-324, 1e-20, 2.0 ** -1022, 1e-19, 1.0, 1e250, np.inf])
    wr, wi = np.empty_like(r2), np.empty_like(r2)
    nf.nf64_weight(_p(r2), ctypes.c_int(len(r2)), ctypes.c_double(1e-20), ctypes.c_double(7.0), _p(wr), _p(wi))
    assert np.all(wr[:4] == 0) and np.all(wi[:4] == 0)
    assert np.all(np.isfinite(wr[:7])) and np.all(np.isfinite(wi[:7]))
    assert np.all(np.hypot(wr[4:7], wi[4:7]) * np.sqrt(r2[4:7]) < 1.0 + 1e-12)
    assert np.isnan(wr[7])


@pytest.mark.gpu
@pytest.mark.parametrize("n,nt,k", [(1, 1, 3.0), (255, 37, 0.0), (4097, 257, 25.0), (20000, 300, -40.0)])
def test_gpu_direct_sizes(n, nt, k):
    """hfmm_direct at tile and chunk edges and k < 0 against the C oracle (the bound of the
    FP64 sum's own test, 1e-13)."""
    import hfmm0_amd
    from oracle import direct as D
    print(f"case: direct N={n} targets={nt} k={k}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(size=(n, 3))
    q = rng.normal(size=n) + 1j * rng.normal(size=n)
    idx = np.sort(rng.choice(n, min(nt, n), replace=False))
    got = hfmm0_amd.direct(x, q, k, idx)
    ref = D.direct_c(x, q, k, idx)
    if n == 1:
        assert got[0] == 0.0
    else:
        assert D.relative_error(got, ref) < 1e-13


@pytest.mark.gpu
@pytest.mark.parametrize("leaf_n", [1, 2, 33, 63, 64, 65, 130])
def test_gpu_fp64_near_field_leaf_sizes(leaf_n):
    """Depth-1 plans (eight leaves, every pair near) against the C oracle: the potential and the
    field of the FP64 near field alone, at target-chunk edges; bound 1e-13 as the direct sum's
    (1e-12 for the field, whose terms grow as r^-2)."""
    import hfmm0_amd
    from oracle import direct as D
    print(f"case: near field, 8 leaves of {leaf_n}", flush=True)
    rng = np.random.default_rng(leaf_n)
    corner = np.array([[i & 1, (i >> 1) & 1, i >> 2] for i in range(8)]) * 0.5
    x = (corner[:, None, :] + rng.uniform(0.0, 0.5, (8, leaf_n, 3))).reshape(-1, 3)
    q = rng.normal(size=len(x)) + 1j * rng.normal(size=len(x))
    st = hfmm0_amd.setup(x, 9.0, p=4, N_max=max(leaf_n, 1), max_depth=1)
    phi = hfmm0_amd.evaluate(st, q)
    phi2, e = hfmm0_amd.evaluate_field(st, q)
    idx = np.arange(len(x))
    ref = D.direct_c(x, q, 9.0, idx)
    assert D.relative_error(phi, ref) < 1e-13 and D.relative_error(phi2, ref) < 1e-13
    eref = D.direct_field_c(x, q, 9.0, idx)
    assert D.relative_error(e, eref) < 1e-12
