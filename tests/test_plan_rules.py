"""Dispatch rules of the plans and pointwise calls (fft_plan.cpp and
pointwise_ops.cpp in ferrum-gpu_amd/csrc), from the code itself: the files are
compiled with g++ beside a small driver and the rules are asked at their edges.  What the rules choose changes no bits, so the GPU
tests that compare results cannot see it."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ferrum-gpu_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

# one rule per line: name, arguments, result
PROGRAM = r"""
#include <stdio.h>
#include <string.h>
#include "fft_plan.hpp"
#include "kernels/tile_geom.h"
#include "pointwise_ops.hpp"
int main() {
    char name[32];
    unsigned long long a, b, c, d;
    while (scanf("%31s %llu %llu %llu %llu", name, &a, &b, &c, &d) == 5) {
        unsigned long long r = 0;
        if (!strcmp(name, "product")) r = fg::product_flags(a) == FG_PASS_LOAD_CACHED;
        else if (!strcmp(name, "convert")) r = fg::convert_flags(a) == FG_PASS_LOAD_CACHED;
        else return 1;
        printf("%llu\n", r);
    }
    return 0;
}
"""

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                                reason="needs g++ and the ROCm headers")


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, exe = d / "rules.cpp", d / "rules"
    src.write_text(PROGRAM)
    # the rules call nothing outside their files, so the rest stays unresolved
    subprocess.run(["g++", "-O0", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}", f"-I{os.path.join(ROOT, 'include')}",
                    f"-I{os.path.join(ROCM, 'include')}", str(src), os.path.join(CSRC, "fft_plan.cpp"), os.path.join(CSRC, "pointwise_ops.cpp"), "-o", str(exe),
                    "-Wl,--unresolved-symbols=ignore-all"], check=True, capture_output=True, text=True, timeout=180)

    def run(calls):
        text = "".join(" ".join(str(v) for v in (list(c) + [0, 0, 0, 0])[:5]) + "\n" for c in calls)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True, timeout=60).stdout.split()
        assert len(out) == len(calls)
        return [int(v) for v in out]

    return run


def test_pointwise_calls_that_load_through_the_caches(ask):
    # n complex elements, 8 n bytes
    assert ask([("product", n) for n in (12 << 17, (13 << 17) - 1, 13 << 17, (40 << 17) - 1, 40 << 17)]) == [0, 0, 1, 1, 0]
    assert ask([("convert", n) for n in ((12 << 17) - 1, 12 << 17, (80 << 17) - 1, 80 << 17)]) == [0, 1, 1, 0]
