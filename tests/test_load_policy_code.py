"""First passes that choose between streamed and cached loads (load_policy,
ferrum-gpu_amd/csrc/kernels/fft_common.hpp) hold both sets of loads in the code
object built from this tree: the compiler may merge two branches whose loads
differ in the cache hint alone, and then every launch loads through the caches
whatever the host asked for."""

import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUNDLE = os.path.join(ROOT, "ferrum-gpu_amd", "csrc", "_build", "fft_kernels.hsaco")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

pytestmark = pytest.mark.skipif(not (os.path.exists(BUNDLE) and os.path.exists(OBJDUMP)),
                                reason="needs the built code object and llvm-objdump")


@pytest.fixture(scope="module")
def loads(tmp_path_factory):
    """Kernel -> (streamed, cached) global load instructions."""
    raw = open(BUNDLE, "rb").read()
    elf = raw
    if raw.startswith(b"__CLANG_OFFLOAD_BUNDLE__"):
        (n,), at = struct.unpack_from("<Q", raw, 24), 32
        for _ in range(n):
            off, size, name_len = struct.unpack_from("<3Q", raw, at)
            name = raw[at + 24:at + 24 + name_len]
            at += 24 + name_len
            if b"gfx950" in name:
                elf = raw[off:off + size]
    path = tmp_path_factory.mktemp("code") / "fft_kernels.elf"
    path.write_bytes(elf)
    text = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
    counts, kernel = {}, None
    for line in text.splitlines():
        m = re.match(r"^[0-9a-f]+ <(\w+)>:", line)
        if m:
            kernel = counts.setdefault(m[1], [0, 0])
        elif kernel is not None and "global_load_" in line:
            kernel[0 if re.search(r"\bnt\b", line) else 1] += 1
    return counts


def _first_pass_kernels(counts):
    """The kernels whose first loads take either policy: single-pass ones in
    both layouts, 2D row passes (interleaved _sc, split _si)."""
    return [k for k in counts if re.fullmatch(r"fg_fft_n\d+(_lat)?(_split)?|fg_fft_n\d+_(sc|si)|fg_fft2d_l\d+_\d+(_split)?", k)]


def test_every_first_pass_keeps_its_streamed_loads(loads):
    kernels = _first_pass_kernels(loads)
    assert len(kernels) > 60
    for k in kernels:
        streamed, cached = loads[k]
        base = re.sub(r"_(split|si)$", "", k)
        split = base != k
        # one load per element and thread, two on the split layout
        want = loads[base][0] * (2 if split else 1)
        assert streamed == want > 0, (k, streamed, want)
        assert cached >= streamed, (k, cached, streamed)  # the other branch's (and the twiddle tables')
