"""Checks of the kernels' sources that no run can make: an ordering that is
missing in the source can still hold in one compiler's output."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "decide_amd", "csrc")


def test_wave_barriers_order_memory():
    """__builtin_amdgcn_wave_barrier is no memory operation: the compiler may move
    LDS accesses across it. Each one stands between a release and an acquire
    fence of the wave."""
    found = 0
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".hpp")):
            continue
        with open(os.path.join(CSRC, name)) as f:
            src = re.sub(r"//[^\n]*", "", f.read())
        statements = [s.strip() for s in re.split(r"[;{}]", src)]
        for i, s in enumerate(statements):
            if s != "__builtin_amdgcn_wave_barrier()":
                continue
            found += 1
            assert statements[i - 1] == '__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront")', name
            assert statements[i + 1] == '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront")', name
    assert found, "attention.hip's key-split kernel has them"
