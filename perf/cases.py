"""Performance cases of the FFT path: batched power-of-two C2C complex64
transforms through the package's public entry points (ferrum_gpu.fft,
ferrum_gpu.pointwise).

A case is a dict of plain values:
  api        "plan"   Plan1D / Plan2D.execute on device arrays, out of place
             "split"  Plan.execute_split, real and imaginary f32 arrays
             "filter" forward, spectrum product, normalised inverse: the
                      product and the inverse in place on the spectrum
             "host"   fft_1d_c2c_pow2 / fft_2d_c2c_pow2 on numpy arrays
  log_rows   0 for 1D, else log2 of the image's rows
  log_n      log2 of the transform length (2D: of the image's columns)
  batch      transforms (images) per call
  direction  "forward", "inverse" (normalised) or "roundtrip" (forward, then
             the normalised inverse of its result); "filter": "forward"
"""

from __future__ import annotations

import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferrum-gpu_amd"))
import ferrum_gpu  # noqa: E402

MOST = 1 << 26  # complex elements of the largest case: 512 MiB in, 512 MiB out


def _case(name, api, log_rows, log_n, batch, direction):
    return {"name": name, "api": api, "log_rows": log_rows, "log_n": log_n, "batch": batch, "direction": direction}


def listed():
    return [
        # The smallest calls: short frames transformed and back, bound by
        # latency and launches (256 frames of 256 points, as in the benchmark).
        _case("1d_256x256_roundtrip", "plan", 0, 8, 256, "roundtrip"),
        # Range-Doppler and STFT sized blocks, an odd number of them.
        _case("1d_4096x1023_inverse", "plan", 0, 12, 1023, "inverse"),
        # The benchmark's headline: a large batch of short transforms.
        _case("1d_1024x65536", "plan", 0, 10, 65536, "forward"),
        # Multi-channel recordings: fewer long transforms than the GPU has CUs.
        _case("1d_32768x96_inverse", "plan", 0, 15, 96, "inverse"),
        # A stack of long records.
        _case("1d_2p17x100_inverse", "plan", 0, 17, 100, "inverse"),
        # One long signal on its own.
        _case("1d_2p20x1", "plan", 0, 20, 1, "forward"),
        # The largest 1D length, four signals (as in the benchmark).
        _case("1d_2p24x4", "plan", 0, 24, 4, "forward"),
        # A few camera-sized image tiles.
        _case("2d_512x3", "plan", 9, 9, 3, "forward"),
        # Large images, two at a time (as in the benchmark).
        _case("2d_4096x2", "plan", 12, 12, 2, "forward"),
        # Callers that keep real and imaginary parts apart.
        _case("split_1d_2p18x16", "split", 0, 18, 16, "forward"),
        # Filtering images in the frequency domain, in place on the spectrum.
        _case("filter_2d_1024x3", "filter", 10, 10, 3, "forward"),
        # The numpy call: copies in and out of the GPU included.
        _case("host_1d_1024x512", "host", 0, 10, 512, "forward"),
    ]


def draw(rng):
    """One more case: every length of both ranks, totals spread over their
    logarithm from a few frames to 512 MiB, any batch that gives."""
    api = rng.choice(["plan"] * 6 + ["split", "split", "filter", "host"])
    if rng.random() < 0.55:
        log_rows, log_n = 0, rng.randint(2, 24)
    else:
        log_rows, log_n = rng.randint(4, 12), rng.randint(4, 12)
    direction = "forward" if api == "filter" else rng.choice(["forward", "forward", "inverse", "roundtrip"])
    # a round trip and a filter run two transforms, a host call two copies
    # over the link: less of it costs what the largest listed case does
    top = {"plan": 26.0, "split": 25.0, "filter": 24.5, "host": 22.0}[api]
    if direction == "roundtrip":
        top -= 1.0
    total = 2.0 ** rng.uniform(16.0, top)
    if total < 2.0 ** 20 and api == "plan":
        direction = "roundtrip"  # a single launch of a few frames is too short to time on its own
    batch = max(1, int(total) >> (log_rows + log_n))
    if batch << (log_rows + log_n) > MOST:
        batch = MOST >> (log_rows + log_n)
    return {"api": api, "log_rows": log_rows, "log_n": log_n, "batch": batch, "direction": direction}


def _shape(case):
    if case["log_rows"]:
        return (case["batch"], 1 << case["log_rows"], 1 << case["log_n"])
    return (case["batch"], 1 << case["log_n"])


def _elems(case):
    return case["batch"] << (case["log_rows"] + case["log_n"])


_device = None


def _dev():
    global _device
    if _device is None:
        _device = ferrum_gpu.hip.Device(0)
    return _device


def _signal(case, seed):
    """Samples in [-1, 1), real and imaginary part independent."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.rand(_shape(case) + (2,), generator=g, device="cuda", dtype=torch.float32)
    return torch.view_as_complex(x.mul_(2.0).sub_(1.0))


def _response(case, seed):
    """A filter's frequency response: one per image or transform, magnitude one."""
    g = torch.Generator(device="cuda").manual_seed(seed + 7919)
    phase = torch.rand(_shape(case), generator=g, device="cuda", dtype=torch.float32).mul_(6.2831853)
    return torch.polar(torch.ones_like(phase), phase)


def prepare(case, seed):
    """Inputs, outputs and the plan that a program holds before the call."""
    dev = _dev()
    x = _signal(case, seed)
    s = {"case": case}
    if case["api"] == "host":
        s["x"] = x.cpu().numpy()
        if not case["log_rows"]:
            s["x"] = s["x"].reshape(-1)
        return s
    if case["log_rows"]:
        s["plan"] = ferrum_gpu.fft.Plan2D(case["log_rows"], case["batch"], dev, log_cols=case["log_n"])
    else:
        s["plan"] = ferrum_gpu.fft.Plan1D(case["log_n"], case["batch"], dev)
    if case["api"] == "split":
        s["re"], s["im"] = x.real.contiguous(), x.imag.contiguous()
        s["out_re"], s["out_im"] = torch.empty_like(s["re"]), torch.empty_like(s["im"])
        if case["direction"] == "roundtrip":
            s["back_re"], s["back_im"] = torch.empty_like(s["re"]), torch.empty_like(s["im"])
    else:
        s["x"], s["y"] = x, torch.empty_like(x)
        if case["direction"] == "roundtrip":
            s["back"] = torch.empty_like(x)
        if case["api"] == "filter":
            s["h"] = _response(case, seed)
    torch.cuda.synchronize()  # the plan's stream is not torch's
    return s


def run(s):
    """One pass on the device's default stream (host calls: until they return)."""
    case = s["case"]
    d = case["direction"]
    if case["api"] == "host":
        first = "inverse" if d == "inverse" else "forward"
        y = _host_call(case, s["x"], first)
        return [y, _host_call(case, y, "inverse")] if d == "roundtrip" else y
    plan = s["plan"]
    if case["api"] == "filter":
        plan.execute(s["x"], s["y"], "forward")
        ferrum_gpu.pointwise.cmul(_dev(), s["y"], s["h"], s["y"], s["y"].numel())
        plan.execute(s["y"], s["y"], "inverse", normalize=True)
        return s["y"]
    if case["api"] == "split":
        if d == "inverse":
            plan.execute_split(s["re"], s["im"], s["out_re"], s["out_im"], "inverse", normalize=True)
        else:
            plan.execute_split(s["re"], s["im"], s["out_re"], s["out_im"], "forward")
        if d == "roundtrip":
            plan.execute_split(s["out_re"], s["out_im"], s["back_re"], s["back_im"], "inverse", normalize=True)
            return [s["out_re"], s["out_im"], s["back_re"], s["back_im"]]
        return [s["out_re"], s["out_im"]]
    if d == "inverse":
        plan.execute(s["x"], s["y"], "inverse", normalize=True)
    else:
        plan.execute(s["x"], s["y"], "forward")
    if d == "roundtrip":
        plan.execute(s["y"], s["back"], "inverse", normalize=True)
        return [s["y"], s["back"]]
    return s["y"]


def _host_call(case, x, direction):
    dev = _dev()
    norm = direction == "inverse"
    if not case["log_rows"]:
        return ferrum_gpu.fft.fft_1d_c2c_pow2(x, case["log_n"], direction, norm, dev)
    if case["log_rows"] == case["log_n"]:
        return ferrum_gpu.fft.fft_2d_c2c_pow2(x, case["log_n"], direction, norm, dev)
    return ferrum_gpu.fft.fft2_c2c_pow2(x, direction, norm, dev)


def exact(case, seed):
    """The same values from torch's CPU transforms in complex128."""
    x = _signal(case, seed).cpu().to(torch.complex128)
    dims = (-2, -1) if case["log_rows"] else (-1,)
    d = case["direction"]
    y = torch.fft.ifftn(x, dim=dims) if d == "inverse" else torch.fft.fftn(x, dim=dims)
    if case["api"] == "filter":
        return torch.fft.ifftn(y * _response(case, seed).cpu().to(torch.complex128), dim=dims)
    if case["api"] == "split":
        out = [y.real.contiguous(), y.imag.contiguous()]
        return out + [x.real.contiguous(), x.imag.contiguous()] if d == "roundtrip" else out
    if case["api"] == "host":
        shape = (-1,) if not case["log_rows"] else _shape(case)
        y, x = y.reshape(shape).numpy(), x.reshape(shape).numpy()
    return [y, x] if d == "roundtrip" else y


def work(case):
    """One read and one write of the data per transform; a filter also reads
    the spectrum and the response and writes the product."""
    n = _elems(case)
    log_points = case["log_rows"] + case["log_n"]
    transforms = 2 if case["direction"] == "roundtrip" or case["api"] == "filter" else 1
    byte = 16 * n * transforms + (24 * n if case["api"] == "filter" else 0)
    flop = 5 * n * log_points * transforms + (6 * n if case["api"] == "filter" else 0)
    return {"bytes": byte, "flops": flop}


def tolerance(case):
    """Four times the relative 2-norm errors measured against exact(): 0.9e-7
    to 1.5e-7 for 1D transforms of up to 32768 points, 1.3e-7 to 1.9e-7 for
    2D ones, 4.7e-7 to 7.2e-7 for longer 1D transforms, whose passes form
    their twiddles by a recurrence in f32; the errors of a transform and of
    its way back add up."""
    rel = 8e-7 if case["log_rows"] else 6e-7 if case["log_n"] <= 15 else 3e-6
    two = case["direction"] == "roundtrip" or case["api"] == "filter"
    return {"rel": 2 * rel if two else rel}
