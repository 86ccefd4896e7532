"""Device memory of a batch: the partial sums of the split M2L blocks are the batch's, in one buffer of
at most 4 GiB, and a plan of a batch takes its own only when it is first evaluated alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MIB = 2 ** 20


def _used():
    import torch
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return (total - free) / MIB


def _problems(n_problems, n, seed=0):
    rng = np.random.default_rng(seed)
    return [(rng.uniform(size=(n, 3)), rng.normal(size=n) + 1j * rng.normal(size=n)) for _ in range(n_problems)]


def test_plans_of_a_batch_hold_no_partial_sums():
    """64 problems of 20000 points in FP64, p = 10: the expansions, their (S, D) copies and the lists
    are some 25 MiB a problem, the partial sums of a plan's own evaluate another 40."""
    import hfmm0_amd as hf
    from hfmm0_amd.batch import Batch
    probs = _problems(64, 20000)
    hf.evaluate(hf.setup(*probs[0][:1], 5.0, p=10, N_max=64), probs[0][1])   # kernels and tables loaded
    u = _used()
    B = Batch([x for x, _ in probs], [5.0] * len(probs), p=10, N_max=64)
    plans = _used() - u
    print(f"case: batch of 64 in FP64: plans {plans:.0f} MiB", flush=True)
    assert plans < 64 * 45
    out = B.evaluate([q for _, q in probs])
    batch = _used() - u - plans
    print(f"  batch evaluate {batch:.0f} MiB", flush=True)
    alone = hf.evaluate(B.plan(1), probs[1][1])            # takes its own partial sums now
    assert np.linalg.norm(alone - out[1]) <= 1e-13 * np.linalg.norm(alone)
    again = B.evaluate([q for _, q in probs])
    assert np.linalg.norm(again[1] - out[1]) <= 1e-13 * np.linalg.norm(alone)
    B.close()


def test_partial_sums_are_bounded():
    """160 mixed problems of 6000 points at p = 15 would leave more than 4 GiB of partial sums in one
    launch: several launches, with each problem's own result.  (FP64 atomics of coarse M2M levels leave
    the order of some sums open: 1e-12 is far above what that moves.)"""
    import hfmm0_amd as hf
    from hfmm0_amd.batch import Batch
    n, m = 6000, 160
    probs = _problems(m, n, 1)
    kw = dict(p=15, N_max=12, precision="mixed")
    u = _used()
    B = Batch([x for x, _ in probs], [5.0] * m, **kw)
    plans = _used() - u
    out = B.evaluate([q for _, q in probs])
    batch = _used() - u - plans - m * n * 32 / MIB    # less the call's device copies of q and phi
    print(f"case: batch of {m} mixed at p = 15: plans {plans:.0f} MiB, evaluate {batch:.0f} MiB", flush=True)
    assert batch < 4096 + 512
    for i in (0, m // 2, m - 1):
        st = hf.setup(probs[i][0], 5.0, **kw)
        alone = hf.evaluate(st, probs[i][1])
        st.close()
        assert np.linalg.norm(out[i] - alone) <= 1e-12 * np.linalg.norm(alone)
    B.close()
