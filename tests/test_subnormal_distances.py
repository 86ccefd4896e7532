"""FP64 pairs closer than 1.5e-154, whose r^2 is a subnormal number: the weight is that of the r^2
given.  1/r of the host build is off by at most 2 ulp (the bound of normal r^2); r carries the rounding
of its residual to 2^-1075, a relative 2^-1075 / (2 r^2), which only its phase k r sees."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def nf(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("nf") / "libnf64.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-march=x86-64-v3", "-ffp-contract=off", "-fPIC", "-shared",
                    os.path.join(HERE, "native", "nearfield64_host.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("k", [0.0, 7.0])
def test_weight(nf, k):
    r2 = np.concatenate([np.geomspace(5e-324, 2.0 ** -1022, 2001), [2.0 ** -1022, 1e-300, 1.0]])
    wr, wi = np.empty_like(r2), np.empty_like(r2)
    p = [a.ctypes.data_as(ctypes.c_void_p) for a in (r2, wr, wi)]
    nf.nf64_weight(p[0], ctypes.c_int(len(r2)), ctypes.c_double(0.0), ctypes.c_double(k), p[1], p[2])
    r = np.sqrt(r2.astype(np.longdouble))
    err = np.hypot((wr * r - np.cos(k * r)).astype(float), (wi * r - np.sin(k * r)).astype(float))
    assert np.max(err) <= 4 * 2.0 ** -52 + 1e-15


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-150, 1e-155, 1e-157, 1e-160])
def test_gpu_direct(scale):
    """Eight points `scale` apart: 1/r to the bits that r^2 holds (2^-1075 / r^2, at least 2^-50)."""
    import hfmm0_amd
    print(f"case: direct sum of points {scale} apart", flush=True)
    x = np.array([[i & 1, (i >> 1) & 1, i >> 2] for i in range(8)]) * scale
    q = np.arange(1.0, 9.0)
    got = hfmm0_amd.direct(x, q, 3.0, np.arange(8))
    d = x[:, None].astype(np.longdouble) - x[None]
    r = np.sqrt((d * d).sum(axis=2))
    np.fill_diagonal(r, 1.0)
    w = 1.0 / r
    np.fill_diagonal(w, 0.0)
    ref = (w @ q).astype(float)
    assert np.linalg.norm(got.real - ref) <= (2.0 ** -50 + 2.0 ** -1074 / scale ** 2) * np.linalg.norm(ref)
