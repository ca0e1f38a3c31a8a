"""What a kernel's source has to spell out because no run shows its absence."""
import glob
import os
import re
import subprocess

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


HANDED_OFF = r"""
#include <stdio.h>
#define __host__
#define __device__
#include "handed_off.h"
static int nan16(uint32_t h) { return (h & 0x7C00u) == 0x7C00u && (h & 0x3FFu); }
static int nan32(uint32_t w) { return (w & 0x7F800000u) == 0x7F800000u && (w & 0x7FFFFFu); }
int main() {
    long bad = 0;
    for (uint64_t i = 0; i < 1ull << 32; i++) {
        const uint32_t w = (uint32_t)i, two = fh::written2(w), one = fh::written1(w);
        bad += two == fh::NOT_YET || one == fh::NOT_YET;
        if (two != w)
            for (int half = 0; half < 32; half += 16) {
                const uint32_t from = w >> half & 0xFFFFu, to = two >> half & 0xFFFFu;
                bad += from != to && !(from == 0xFFFFu && nan16(to) && (from ^ to) == 0x8000u);
            }
        bad += one != w && !(w == ~0u && nan32(one) && (one ^ w) == 0x80000000u);
    }
    printf("%ld", bad);
}
"""


def test_a_number_handed_off_is_never_unwritten(tmp_path):
    """Every word: what is stored in place of it is not the mark of an unwritten one, and is it but for the sign of the NaN of all ones."""
    (tmp_path / "t.cc").write_text(HANDED_OFF)
    subprocess.check_call(["g++", "-O2", "-I", CSRC, str(tmp_path / "t.cc"), "-o", str(tmp_path / "t")])
    assert subprocess.check_output([str(tmp_path / "t")], timeout=110) == b"0"
