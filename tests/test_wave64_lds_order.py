"""The rows of m2l_wave64.hip's LDS columns pass between lanes of a wave, so every point where a lane
reads a row that another wrote (or writes one that another read or wrote) needs a wavefront fence:
without it the compiler sees addresses of one lane, a constant apart, and may reorder them.  Counted
in the kernels' IR as the front end makes it, before any pass."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hfmm0_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def calls(tmp_path_factory):
    """function -> (its calls in the module, its fences of wavefront scope)"""
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("ir") / "wave64.ll")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "--offload-device-only", "-S", "-emit-llvm",
                    "-Xclang", "-disable-llvm-passes", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    os.path.join(CSRC, "m2l_wave64.hip"), "-o", out], check=True, stderr=subprocess.DEVNULL)
    fns, cur = {}, None
    define = re.compile(r'^define .*?@("[^"]+"|[\w.$]+)\(')
    call = re.compile(r'\bcall .*?@("[^"]+"|[\w.$]+)\(')
    with open(out) as f:
        for line in f:
            m = define.match(line)
            if m:
                cur = fns[m.group(1)] = [[], 0]
            elif cur is not None:
                if line.startswith("}"):
                    cur = None
                elif re.match(r'\s*fence syncscope\("wavefront"\) acq_rel', line):
                    cur[1] += 1
                else:
                    m = call.search(line)
                    if m:
                        cur[0].append(m.group(1))
    return fns


@pytest.mark.parametrize("p", range(2, 15))
def test_fences(calls, p):
    memo = {}

    def fences(fn):   # executed by a call of fn, straight-line code
        if fn not in calls:
            return 0
        if fn not in memo:
            memo[fn] = calls[fn][1] + sum(fences(c) for c in calls[fn][0])
        return memo[fn]

    kernels = [f for f in calls if re.search(r"wave64(_batch)?_kernelILi%dE" % p, f)]
    assert len(kernels) == 2
    # once after the columns are cleared; per half: before the gather, after the last register of every
    # degree that it does not fill (the next degree overwrites what lies past its rows), after each of the
    # three stages, and after the gather where degree p fills its registers (no fence of its own)
    overflow = sum(n % 4 != 3 for n in range(p + 1))
    need = 1 + 2 * (1 + overflow + 3 + (1 if p % 4 == 3 else 0))
    for f in kernels:
        assert fences(f) >= need, (f, fences(f), need)
