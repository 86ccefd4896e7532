"""A charge that is not finite reaches every other point and not its own: the pair of a point with
itself (and with a coincident point) contributes nothing whatever the charge, in the FP64 near field,
with the field, and in both direct sums.  The values at those points are the sums over the other
charges; the rest are not finite.

Bounds as for finite charges: 1e-13 of the l2 norm, 1e-12 for the field."""
import ctypes

import numpy as np
import pytest

from oracle import direct as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hf():
    import hfmm0_amd
    return hfmm0_amd


def _cloud(n, seed):
    rng = np.random.default_rng(seed + n)
    x, q = rng.uniform(size=(n, 3)), rng.normal(size=n) + 1j * rng.normal(size=n)
    return x, q


def _noalloc(x, q, k, idx):
    import torch
    from hfmm0_amd import _lib as L
    xd, qd, td = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (x, q, idx.astype(np.int64)))
    od = torch.zeros(len(idx), dtype=torch.complex128, device="cuda")
    torch.cuda.synchronize()
    L.check(L.lib().hfmm_direct_noalloc(ctypes.c_void_p(xd.data_ptr()), len(x), ctypes.c_void_p(qd.data_ptr()),
                                        float(k), ctypes.c_void_p(td.data_ptr()), len(idx),
                                        ctypes.c_void_p(od.data_ptr()), None))
    torch.cuda.synchronize()
    return od.cpu().numpy()


BAD = [np.nan, np.inf, complex(0.0, -np.inf), complex(1e308, 1e308)]


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("n,k", [(5, 3.0), (130, 0.0), (300, -7.0), (1000, 25.0)])
def test_own_point(hf, n, k, bad):
    print(f"case: charge {bad} at one of {n} points, k={k}", flush=True)
    x, q = _cloud(n, 1)
    at = n // 3
    x[n - 1] = x[at]                       # a coincident point
    own = np.array([at, n - 1])
    rest = q.copy()
    rest[own] = 0.0
    ref = D.direct_c(x, rest, k, own)
    eref = D.direct_field_c(x, rest, k, own)
    q[at] = bad
    q[n - 1] = bad
    others = np.setdiff1d(np.arange(n), own)
    st = hf.setup(x, k, p=4, N_max=2048)   # one leaf: the near field alone
    phi, e = hf.evaluate_field(st, q)
    values = {"near field": hf.evaluate(st, q), "with field": phi, "direct": hf.direct(x, q, k, np.arange(n)),
              "direct, no allocation": _noalloc(x, q, k, np.arange(n))}
    for name, v in values.items():
        print(f"  {name}: own {v[own]} reference {ref}", flush=True)
        assert np.isfinite(v[own]).all(), name
        assert np.linalg.norm(v[own] - ref) <= 1e-13 * np.linalg.norm(ref), name
        if not np.isfinite(bad):
            assert not np.isfinite(v[others]).any(), name
    assert np.isfinite(e[own]).all()
    assert np.linalg.norm(e[own] - eref) <= 1e-12 * np.linalg.norm(eref)
