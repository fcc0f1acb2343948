"""1D last passes on the GPU: every row-wise tile kernel (128, 256, 512 and
1024 points) at one transform, at a ragged batch and with two chunks in
flight, forward and normalised inverse, against the oracle."""

import numpy as np
import pytest

import oracle
from conftest import normal_c64, rel_l2

pytestmark = pytest.mark.gpu

# Four times the relative 2-norm error of these lengths against 64 bits
# (7.2e-7 at 2^24, the longest twiddle recurrences) and the oracle's own f32
# error beside it (up to 1e-6 at 2^22).
TOL = 5e-6

CASES = [(16, 1, None), (17, 1, None), (17, 5, 4 << 20), (18, 1, None), (18, 3, None), (18, 5, 8 << 20), (19, 1, None),
         (19, 3, 8 << 20), (20, 1, None), (20, 3, 16 << 20), (21, 1, None), (22, 1, None)]


@pytest.mark.parametrize("log_n,batch,limit", CASES)
def test_last_pass_against_the_oracle(gpu_device, log_n, batch, limit):
    import ferrum_gpu
    from ferrum_gpu.hip import DeviceBuffer

    saved = ferrum_gpu.fft.get_chunk_bytes()
    if limit:
        ferrum_gpu.fft.set_chunk_bytes(limit)
    try:
        plan = ferrum_gpu.fft.Plan1D(log_n, batch, gpu_device)
    finally:
        ferrum_gpu.fft.set_chunk_bytes(saved)
    d = plan.describe()
    print(f"[case] log_n={log_n} batch={batch} {plan.kernel_names()} {d}", flush=True)
    assert d["streams"] == (2 if limit else 1)
    x = normal_c64(np.random.default_rng(1200 + log_n + batch), batch << log_n)
    a, b = DeviceBuffer(gpu_device, plan.nbytes), DeviceBuffer(gpu_device, plan.nbytes)
    a.copy_from_host(x)
    for direction, normalize in (("forward", False), ("inverse", True)):
        plan.execute(a, b, direction, normalize)
        gpu_device.sync()
        got = b.copy_to_host(np.empty_like(x))
        assert rel_l2(got, oracle.fft_1d(x, log_n, direction, normalize, threads=8)) <= TOL
    plan.destroy()
