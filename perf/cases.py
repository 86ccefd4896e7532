"""Work that users of this library have it do, for timing and for comparing two builds.

Every case is one call through a public entry point on inputs made from a seed: potentials at
all points (`evaluate`, `evaluate_device`, and `hfmm_evaluate_typed` of the C ABI for a
device-resident complex64 result), the potential with its field (`evaluate_field`), a batch of
problems (`Batch`), and the direct sum at sampled targets (`direct`) that certifies results.
A plan is made once per geometry and evaluated for many charge vectors, so plans belong to the
state.  Results of the plain FP64 form are complex128; the mixed form, whose near field and
translations are FP32, is called with its complex64 result.

`listed()` gives the named cases, `draw(rng)` one more of the same ranges, `prepare(case, seed)`
the state, `run(state)` one pass, `work(case)` the bytes and operations that a pass cannot do
without, `exact(case, seed)` the same outputs by the plain direct sum in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

import hfmm0_amd
from hfmm0_amd import _lib
from hfmm0_amd.api import torch_charge_code
from hfmm0_amd.batch import Batch
from hfmm0_amd.learned import degree_floor
from hfmm0_amd.workloads import P2P_FLOPS_PER_PAIR, f_m2l

# pairs of a direct sum in FP64 that plain torch does in well under 20 seconds
EXACT_PAIRS = 2.0e11


def listed():
    return [
        # The size and leaf of the reference's own harness: a solver's inner iteration on a small
        # scatterer, NumPy in and out, real charges.  Latency and launches are all of it.
        {"name": "harness_640", "call": "evaluate", "n": 640, "k": 3.0, "p": 6, "leaf": 16, "points": "cube",
         "charges": "f64", "precision": "fp64"},
        # The reference-parity configuration: 20k points, k = 10, p = 10, leaves of 64, NumPy in and out.
        {"name": "parity_20k", "call": "evaluate", "n": 20000, "k": 10.0, "p": 10, "leaf": 64, "points": "cube",
         "charges": "c128", "precision": "fp64"},
        # A boundary-element operator in double precision: points on surfaces (W and X lists, uneven
        # leaves), charges resident on the GPU between the steps of an iterative solver.
        {"name": "surface_60k_fp64", "call": "device", "n": 60011, "k": 25.0, "p": 12, "leaf": 64,
         "points": "sphere_clusters", "charges": "c128", "precision": "fp64"},
        # The plain form at the degree that six digits of a volume problem take.
        {"name": "volume_400k_fp64", "call": "device", "n": 400000, "k": 20.0, "p": 14, "leaf": 128,
         "points": "cube", "charges": "c128", "precision": "fp64"},
        # Forces or near-field scans: potential and field, NumPy in and out.
        {"name": "field_40k", "call": "field", "n": 40000, "k": 12.0, "p": 10, "leaf": 64, "points": "cube",
         "charges": "c128", "precision": "fp64"},
        # Many small uneven problems at once (bodies of a multi-scatterer, frequencies of a sweep).
        {"name": "batch_16", "call": "batch", "problems": 16, "n_min": 2000, "n_max": 20000, "k": 25.0, "p": 10,
         "leaf": 64, "points": "ellipsoid", "charges": "c128", "precision": "fp64"},
        # Certifying a result: the direct sum at 4096 sampled targets of the million-point workload.
        {"name": "certify_1m", "call": "direct", "n": 1000000, "k": 40.0, "targets": 4096, "points": "cube",
         "charges": "c128"},
        # Electrostatics (k = 0) with single-precision real charges, three to four digits, NumPy in and out.
        {"name": "coulomb_150k", "call": "evaluate", "n": 150000, "k": 0.0, "p": 7, "leaf": 64, "points": "cube",
         "charges": "f32", "precision": "mixed"},
        # An ordinary mixed-precision evaluate: NumPy in and out, complex64 charges, odd size.
        {"name": "mixed_100k", "call": "evaluate", "n": 100003, "k": 15.0, "p": 11, "leaf": 128, "points": "mixed",
         "charges": "c64", "precision": "mixed"},
        # The adaptive configuration at a size the direct sum can check: sphere and clusters,
        # device-resident, degrees raised on the coarse levels by the high-frequency floor.
        {"name": "surface_300k", "call": "device", "n": 300000, "k": 50.0, "p": 10, "leaf": 128,
         "points": "sphere_clusters", "charges": "c64", "precision": "mixed"},
        # The headline workload: a million points in the cube, k = 40, leaves of 128, the
        # certified per-level degrees of a 1e-6 result, device-resident.
        {"name": "volume_1m", "call": "device", "n": 1000000, "k": 40.0, "p": 18, "p_level": "18,18,14,12,11",
         "leaf": 128, "points": "cube", "charges": "c64", "precision": "mixed"},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    call = rng.choice(["evaluate", "evaluate", "device", "device", "mixed", "mixed", "mixed", "field", "batch",
                       "direct"])
    points = rng.choice(["cube", "cube", "sphere_clusters", "mixed", "ellipsoid"])
    if call == "evaluate":     # plain form, NumPy in and out
        return {"call": call, "n": int(_log(rng, 300, 20000)), "k": round(rng.uniform(0.0, 10.0), 3),
                "p": rng.randint(4, 12), "leaf": rng.choice([16, 32, 64]), "points": points,
                "charges": rng.choice(["f64", "c128"]), "precision": "fp64"}
    if call == "device":       # plain form, device-resident
        return {"call": call, "n": int(_log(rng, 20000, 300000)), "k": round(rng.uniform(2.0, 20.0), 3),
                "p": rng.randint(8, 14), "leaf": rng.choice([64, 128]), "points": points, "charges": "c128",
                "precision": "fp64"}
    if call == "mixed":
        host = rng.random() < 0.4
        return {"call": "evaluate" if host else "device", "n": int(_log(rng, 20000, 150000 if host else 400000)),
                "k": 0.0 if rng.random() < 0.2 else round(rng.uniform(2.0, 40.0), 3), "p": rng.randint(6, 14),
                "leaf": rng.choice([64, 128]), "points": points, "charges": rng.choice(["c64", "c64", "f32"]),
                "precision": "mixed"}
    if call == "field":
        return {"call": call, "n": int(_log(rng, 4000, 40000)), "k": round(rng.uniform(0.5, 12.0), 3),
                "p": rng.randint(6, 11), "leaf": 64, "points": points, "charges": rng.choice(["f64", "c128"]),
                "precision": "fp64"}
    if call == "batch":
        return {"call": call, "problems": rng.randint(4, 16), "n_min": 2000, "n_max": int(_log(rng, 4000, 20000)),
                "k": round(rng.uniform(5.0, 25.0), 3), "p": rng.randint(6, 11), "leaf": rng.choice([64, 128]),
                "points": "ellipsoid", "charges": "c128", "precision": "fp64"}
    return {"call": "direct", "n": int(_log(rng, 60000, 1000000)), "k": round(rng.uniform(0.0, 40.0), 3),
            "targets": rng.randint(200, 4096), "points": points, "charges": "c128"}


# ---- inputs ------------------------------------------------------------------------------

def _points(kind, n, rng):
    def sphere(m):
        v = rng.normal(size=(m, 3))
        return 0.5 + 0.45 * v / np.linalg.norm(v, axis=1, keepdims=True)

    def clusters(m):
        c = rng.uniform(0.1, 0.9, (8, 3))
        return c[rng.integers(0, 8, m)] + rng.normal(scale=0.02, size=(m, 3))

    if kind == "cube":
        return rng.uniform(0.0, 1.0, (n, 3))
    if kind == "ellipsoid":
        axes = rng.uniform(0.2, 0.5, 3)
        v = rng.normal(size=(n, 3))
        v *= (rng.uniform(size=n) ** (1.0 / 3.0) / np.linalg.norm(v, axis=1))[:, None]
        return 0.5 + v * axes
    if kind == "sphere_clusters":
        return np.vstack([sphere(n // 2), clusters(n - n // 2)])
    a = n // 3
    return np.vstack([rng.uniform(0.0, 1.0, (a, 3)), sphere(a), clusters(n - 2 * a)])


def _charges(kind, n, rng):
    q = rng.normal(size=n)
    if kind in ("f64", "f32"):
        return q.astype(np.float32) if kind == "f32" else q
    q = q + 1j * rng.normal(size=n)
    return q.astype(np.complex64) if kind == "c64" else q


def _degrees(case, k):
    """Per-level degrees: the listed ones, or p raised on coarse levels to the high-frequency floor."""
    if case.get("p_level"):
        return [int(v) for v in case["p_level"].split(",")]
    return [max(case["p"], degree_floor(k, 1.0, level)) for level in range(1, 12)]


def _sizes(case):
    """Points of every problem (one, or a batch's sizes spread over their logarithm)."""
    if case["call"] != "batch":
        return [case["n"]]
    m, lo, hi = case["problems"], math.log(case["n_min"]), math.log(case["n_max"])
    return [int(math.exp(lo + (hi - lo) * i / max(1, m - 1))) for i in range(m)]


def _problems(case, seed):
    """(positions, charges, k) of every problem: those of a batch have k up to the case's."""
    rng = np.random.default_rng(seed)
    sizes = _sizes(case)
    out = []
    for i, n in enumerate(sizes):
        x = _points(case["points"], n, rng)
        out.append((x, _charges(case["charges"], n, rng), case["k"] * (i + 1) / len(sizes)))
    return out, rng


def prepare(case, seed):
    probs, rng = _problems(case, seed)
    x, q, k = probs[0]
    call = case["call"]
    if call == "direct":
        return {"call": call, "x": x, "q": q, "k": k, "targets": np.sort(rng.choice(len(x), case["targets"], False))}
    if call == "batch":
        batch = Batch([p[0] for p in probs], [p[2] for p in probs], p=case["p"], N_max=case["leaf"],
                      p_level=[_degrees(case, p[2]) for p in probs], precision=case["precision"])
        qs = [torch.from_numpy(p[1]).cuda() for p in probs]
        return {"call": call, "batch": batch, "q": qs, "out": [torch.empty_like(v) for v in qs]}
    plan = hfmm0_amd.setup(x, k, p=case["p"], N_max=case["leaf"], p_level=_degrees(case, k),
                           precision=case["precision"], tree_device=len(x) > 10000)
    state = {"call": call, "plan": plan, "dtype": np.complex64 if case["precision"] == "mixed" else np.complex128}
    if call == "device":
        state["q"] = torch.from_numpy(q).cuda()
        mixed = case["precision"] == "mixed"
        state["out"] = torch.empty(len(x), dtype=torch.complex64 if mixed else torch.complex128, device="cuda")
    else:
        state["q"] = q
    return state


def run(state):
    call = state["call"]
    if call == "evaluate":
        return hfmm0_amd.evaluate(state["plan"], state["q"], out_dtype=state["dtype"])
    if call == "field":
        return hfmm0_amd.evaluate_field(state["plan"], state["q"])
    if call == "batch":
        return state["batch"].evaluate_device(state["q"], state["out"])
    if call == "direct":
        return hfmm0_amd.direct(state["x"], state["q"], state["k"], state["targets"])
    q, out = state["q"], state["out"]
    if out.dtype == torch.complex128:
        return hfmm0_amd.evaluate_device(state["plan"], q, out)
    # a complex64 result on the GPU: the C ABI's typed evaluate
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.lib().hfmm_evaluate_typed(state["plan"].handle, ctypes.c_void_p(q.data_ptr()),
                                              torch_charge_code(q.dtype), ctypes.c_void_p(out.data_ptr()), _lib.C64,
                                              _lib.DEVICE, ctypes.c_void_p(stream)))
    return out


def work(case):
    """Points and charges read once, results written once; the operations of the algorithm on a
    tree with full leaves: in the cube every box has its 26 neighbours and up to 189 well-separated
    ones; on surfaces about 8 and 27."""
    qb = {"f32": 4, "f64": 8, "c64": 8, "c128": 16}[case["charges"]]
    if case["call"] == "direct":
        return {"bytes": case["n"] * (24 + qb) + case["targets"] * 24,
                "flops": float(case["n"]) * case["targets"] * P2P_FLOPS_PER_PAIR}
    ob = 8 if case["precision"] == "mixed" else 16
    nbytes, flops = 0.0, 0.0
    volume = case["points"] in ("cube", "ellipsoid")
    for i, n in enumerate(_sizes(case)):
        k = case["k"] * (i + 1) / len(_sizes(case))
        pl = _degrees(case, k)
        depth = max(2, math.ceil(math.log(max(n / case["leaf"], 1.0), 8 if volume else 4)))
        for level in range(2, depth + 1):
            side = 2 ** level
            pairs = (4.0 * (3 * side // 2 - 2)) ** 3 - (3.0 * side - 2) ** 3 if volume else 27.0 * 4 ** level
            flops += pairs * f_m2l(pl[min(level, len(pl)) - 1])
        leaves = 8.0 ** depth if volume else 4.0 ** depth
        near = ((3.0 * 2 ** depth - 2) ** 3 if volume else 9.0 * leaves) * (n / leaves) ** 2
        flops += near * P2P_FLOPS_PER_PAIR + 32.0 * n * (pl[min(depth, len(pl)) - 1] + 1) ** 2
        nbytes += n * (24 + qb + ob)
        if case["call"] == "field":
            nbytes += 48.0 * n
            flops += near * 20
    return {"bytes": nbytes, "flops": flops}


# ---- the same outputs by plain sums in 64 bits ---------------------------------------------

def _direct(x, q, k, targets=None, field=False):
    """phi at the targets (all points by default), and E = -grad phi at every point."""
    xs = torch.from_numpy(x).cuda()
    qs = torch.from_numpy(np.asarray(q).astype(np.complex128)).cuda()
    qr, qi = qs.real.contiguous(), qs.imag.contiguous()
    t = xs if targets is None else xs[torch.from_numpy(targets).cuda()]
    phi = torch.zeros(len(t), dtype=torch.complex128, device="cuda")
    e = torch.zeros(len(t), 3, dtype=torch.complex128, device="cuda")
    rows = max(1, int((4 if field else 6) * 10 ** 7) // len(xs))
    for i in range(0, len(t), rows):
        d = [t[i:i + rows, a, None] - xs[None, :, a] for a in range(3)]
        r2 = d[0] * d[0]
        r2.addcmul_(d[1], d[1]).addcmul_(d[2], d[2])
        if not field:
            del d
        r = r2.sqrt_()
        w = torch.where(r > 0, 1.0 / r, 0.0)
        kr = r.mul_(k)
        c, s = torch.cos(kr) * w, torch.sin(kr) * w
        phi[i:i + rows] = torch.complex(c @ qr - s @ qi, c @ qi + s @ qr)
        if field:      # E = sum (x - y)(1 - i k r) e^{ikr} / r^3 q
            fr, fi = (c + kr * s) * w * w, (s - kr * c) * w * w
            for a in range(3):
                gr, gi = fr * d[a], fi * d[a]
                e[i:i + rows, a] = torch.complex(gr @ qr - gi @ qi, gr @ qi + gi @ qr)
    return (phi, e) if field else phi


def exact(case, seed):
    probs, rng = _problems(case, seed)
    x, q, k = probs[0]
    if case["call"] == "direct":
        targets = np.sort(rng.choice(len(x), case["targets"], False))
        return _direct(x, q, k, targets)
    if sum(float(n) ** 2 for n in _sizes(case)) > EXACT_PAIRS:
        return None
    if case["call"] == "field":
        return _direct(x, q, k, field=True)
    if case["call"] == "batch":
        return [_direct(*p) for p in probs]
    phi = _direct(x, q, k)
    return phi.to(torch.complex64) if case["precision"] == "mixed" else phi
