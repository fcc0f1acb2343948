"""Dispatch rules of the plans (ferrum-gpu_amd/csrc/fft_plan.cpp), from the code
itself: the file is compiled with g++ beside a small driver and the rules are
asked at their edges.  What the rules choose changes no bits, so the GPU
tests that compare results cannot see it."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ferrum-gpu_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
MIB = 1 << 20

# one rule per line: name, arguments, result
PROGRAM = r"""
#include <stdio.h>
#include <string.h>
#include "fft_plan.hpp"
int main() {
    char name[32];
    unsigned long long a, b, c, d;
    while (scanf("%31s %llu %llu %llu %llu", name, &a, &b, &c, &d) == 5) {
        unsigned long long r = 0;
        if (!strcmp(name, "single")) r = fg::single_pass_loads_cached(a, b, c);
        else if (!strcmp(name, "image")) r = fg::image_loads_cached(a, b);
        else if (!strcmp(name, "rows")) r = fg::row_pass_loads_cached(a);
        else if (!strcmp(name, "columns")) r = fg::column_pass_loads_cached(a, b, c, d);
        else if (!strcmp(name, "split_narrow")) r = fg::split_narrow_limit(a);
        else if (!strcmp(name, "makes_two")) r = fg::makes_two_chunks(a, b, c);
        else if (!strcmp(name, "runs_two")) r = fg::runs_two_chunks(a, b, c);
        else if (!strcmp(name, "narrow")) r = fg::narrow_width(a, b, c, d);
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
    # the rules call nothing outside their file, so the rest stays unresolved
    subprocess.run(["g++", "-O0", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}", f"-I{os.path.join(ROOT, 'include')}",
                    f"-I{os.path.join(ROCM, 'include')}", str(src), os.path.join(CSRC, "fft_plan.cpp"), "-o", str(exe),
                    "-Wl,--unresolved-symbols=ignore-all"], check=True, capture_output=True, text=True, timeout=180)

    def run(calls):
        text = "".join(" ".join(str(v) for v in (list(c) + [0, 0, 0, 0])[:5]) + "\n" for c in calls)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True, timeout=60).stdout.split()
        assert len(out) == len(calls)
        return [int(v) for v in out]

    return run


def _edges(ask, rule, ranges, *last):
    """ranges: arguments -> (above, up to) in bytes, the inputs that load
    through the caches; last: the rule's arguments after the size."""
    for args, (above, upto) in ranges.items():
        sizes = [above, above + 8, upto, upto + 8] if above else [8, upto, upto + 8]
        want = [0, 1, 1, 0] if above else [1, 1, 0]
        assert ask([(rule, *args, s, *last) for s in sizes]) == want, (rule, args)


def test_first_passes_that_load_through_the_caches(ask):
    for n, upto in [(n, 44) for n in (2, 3, 4, 5, 6, 10)] + [(13, 16), (14, 16), (15, 16)]:
        _edges(ask, "single", {(n,): (0, upto * MIB)})
    for n, top in ((7, 24), (8, 28), (9, 30), (11, 36), (12, 32)):  # streamed between 12 MiB and top
        _edges(ask, "single", {(n,): (0, 12 * MIB)})
        _edges(ask, "single", {(n,): (top * MIB, 44 * MIB)})
    _edges(ask, "image", {(p,): (0, 24 * MIB) for p in (8, 9, 10)})
    _edges(ask, "image", {(p,): (0, 12 * MIB) for p in (11, 12, 13)})
    _edges(ask, "image", {(14,): (0, 20 * MIB)})
    _edges(ask, "rows", {(): (0, 40 * MIB)})
    _edges(ask, "columns", {(16, 32): (0, 56 * MIB), (17, 8): (0, 32 * MIB), (17, 16): (0, 56 * MIB), (18, 16): (0, 80 * MIB),
                            (20, 16): (0, 80 * MIB), (21, 16): (0, 56 * MIB), (24, 32): (0, 56 * MIB)})


def test_split_inputs_have_limits_of_their_own(ask):
    limits = {2: 44, 3: 44, 4: 44, 5: 44, 9: 64, 11: 64, 12: 64, 13: 24, 14: 24, 15: 32}
    _edges(ask, "single", {(n,): (0, limits[n] * MIB) for n in limits}, 1)
    _edges(ask, "single", {(10,): (0, 12 * MIB)}, 1)  # streamed up to 20 MiB
    _edges(ask, "single", {(10,): (20 * MIB, 64 * MIB)}, 1)
    assert all(ask([("single", n, s, 1) for n in (6, 7, 8) for s in (8, MIB, 4096 * MIB)]))  # no limit
    _edges(ask, "columns", {(16, 32): (0, 56 * MIB), (17, 8): (0, 32 * MIB), (17, 16): (0, 56 * MIB), (18, 16): (0, 56 * MIB),
                            (19, 16): (0, 80 * MIB), (20, 16): (0, 80 * MIB), (21, 16): (0, 56 * MIB)}, 1)
    assert ask([("split_narrow", log_l) for log_l in (7, 8, 9, 10)]) == [24 * MIB, 24 * MIB, 24 * MIB, 16 * MIB]


def test_two_chunks_run_at_once_from_a_batch_of_the_limit(ask):
    # unit, batch, limit -> (takes set_streams(2), runs two chunks at a time)
    cases = {(MIB, 128, 256 * MIB): (0, 0), (MIB, 129, 256 * MIB): (1, 0), (MIB, 255, 256 * MIB): (1, 0),
             (MIB, 256, 256 * MIB): (1, 1), (128 * MIB, 1, 256 * MIB): (0, 0), (128 * MIB, 2, 256 * MIB): (1, 1),
             (3 * MIB, 5, 4 * MIB): (0, 0), (MIB, 7, 0): (0, 0), (8 * MIB, 7, 4 * MIB): (0, 0),
             (1 << 40, (1 << 40) - 1, 2**63): (1, 1)}  # unit * batch beyond 2^64
    assert ask([("makes_two", *c) for c in cases]) == [m for m, _ in cases.values()]
    assert ask([("runs_two", *c) for c in cases]) == [r for _, r in cases.values()]


# (log2 points, own columns, tiles per transform or image) -> transforms up to
# which a launch on 256 CUs takes 4, 8, 16 columns (None: never)
NARROW = {(8, 32, 8): (4, 32, 64), (8, 32, 16): (2, 16, 32), (9, 8, 32): (4, None, None), (8, 32, 32): (1, 8, 16),
          (10, 16, 16): (4, 16, None), (9, 16, 64): (1, 8, None), (10, 16, 32): (2, 8, None), (10, 16, 64): (1, 4, None),
          (7, 64, 256): (None, None, 1), (8, 32, 512): (None, None, 1), (7, 64, 16): (None, 8, 16), (9, 16, 32): (2, 16, None),
          (11, 8, 2): (64, None, None), (12, 8, 8): (16, None, None)}


def test_launches_short_of_workgroups_are_narrowed(ask):
    for (log_l, g, tiles), limits in NARROW.items():
        edges = [(w, n) for w, n in zip((4, 8, 16), limits) if n]
        calls, want = [], []
        for i, (w, n) in enumerate(edges):
            calls += [("narrow", log_l, g, tiles * n, 256), ("narrow", log_l, g, tiles * (n + 1), 256)]
            above = [v for v, m in edges[i + 1:] if m >= n + 1]
            want += [w, above[0] if above else 0]
        assert ask(calls) == want, (log_l, g, tiles)


def test_narrow_forms_fit_their_kernels(ask):
    # every width the rule can give: one that the kernel has (tile_narrows in
    # kernels/fft_tile.hpp), a whole wave, no more threads than the kernel's bound
    for log_l, g, per_thread in ((7, 64, 32), (8, 32, 32), (8, 16, 32), (9, 16, 32), (10, 16, 32), (11, 8, 32), (12, 8, 32), (9, 8, 16)):
        got = set(ask([("narrow", log_l, g, t, cu) for t in list(range(1, 300)) + [512, 1024, 4096] for cu in (1, 32, 256, 304)]))
        for w in got - {0}:
            threads = (w << log_l) // 16
            assert w in (4, 8, 16) and w < g and (log_l, g) != (8, 16)
            assert threads % 64 == 0 and 64 <= threads <= (g << log_l) // per_thread
            # the launch steps tiles by g / w of the pass's own (FftPlan::run)
            assert g % w == 0
