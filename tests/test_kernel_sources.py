"""What a kernel's source has to spell out because no run shows its absence."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferrum-infer-rs_amd", "csrc")
COPY, BARRIER = "__builtin_amdgcn_global_load_lds", re.compile(r"__syncthreads\(\)|s_barrier")


def copying_kernels():
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip"))):
        with open(path, encoding="utf-8") as f:
            for body in re.split(r"^(?=__global__)", f.read(), flags=re.M)[1:]:
                if COPY in body:
                    yield pytest.param(body, id=re.search(r"(\w+)\(", re.sub(r"__launch_bounds__\([^\n]*?\) void", "", body)).group(1))


@pytest.mark.parametrize("body", copying_kernels())
def test_copies_to_lds_are_waited_for_by_name(body):
    """Rows copied straight to LDS are read by other waves: a barrier orders the waves, not their outstanding copies."""
    after = body[body.index(COPY):]
    first = BARRIER.search(after)
    assert first and "waitcnt" in after[:first.end()], body[:120]
