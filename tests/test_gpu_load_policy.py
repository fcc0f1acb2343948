"""First passes that load their input through the caches (loads_cached,
ferrum-gpu_amd/csrc/fft_plan.cpp): a batch below the limit gives the bits of
the same transforms at the head of a batch above it, in both layouts, and
agrees with numpy in double precision; ragged last workgroups included."""

import numpy as np
import pytest

from conftest import normal_c64, rel_l2

pytestmark = pytest.mark.gpu

MIB = 1 << 20

# f32 transforms of up to 2^20 points, no twiddle recurrence: four times the
# 1.9e-7 measured against 64 bits.
TOL = 8e-7

# (log_rows, log_n, MiB below, MiB above): below is large enough for the
# throughput kernels (the latency ones of 256, 1024 and 4096 points have
# another radix list).
CASES = [(0, n, 17, 82) for n in range(2, 13)] + [(0, n, 12, 18) for n in (13, 14, 15)] + \
    [(4, 4, 9, 82), (4, 6, 9, 82), (5, 5, 9, 82), (5, 6, 9, 82), (6, 6, 9, 82), (7, 7, 9, 82), (4, 10, 9, 82),
     (6, 9, 40, 66), (10, 10, 40, 72)]


@pytest.mark.parametrize("log_rows,log_n,below,above", CASES)
def test_cached_and_streamed_loads_give_the_same_bits(gpu_device, log_rows, log_n, below, above):
    import ferrum_gpu
    from ferrum_gpu.hip import DeviceBuffer

    unit = 8 << (log_rows + log_n)
    small, big = below * MIB // unit - (1 if log_rows + log_n < 16 else 0), above * MIB // unit + 1
    n_small, n_big = small << (log_rows + log_n), big << (log_rows + log_n)
    print(f"[case] log_rows={log_rows} log_n={log_n} batches {small} and {big}", flush=True)

    def plan(batch):
        if log_rows:
            return ferrum_gpu.fft.Plan2D(log_rows, batch, gpu_device, log_cols=log_n)
        return ferrum_gpu.fft.Plan1D(log_n, batch, gpu_device)

    x = normal_c64(np.random.default_rng(1500 + log_rows + log_n), n_big)
    src, dst = DeviceBuffer(gpu_device, 8 * n_big), DeviceBuffer(gpu_device, 8 * n_big)
    re, im = DeviceBuffer(gpu_device, 4 * n_big), DeviceBuffer(gpu_device, 4 * n_big)
    o_re, o_im = DeviceBuffer(gpu_device, 4 * n_big), DeviceBuffer(gpu_device, 4 * n_big)
    src.copy_from_host(x)
    re.copy_from_host(np.ascontiguousarray(x.real))
    im.copy_from_host(np.ascontiguousarray(x.imag))
    p_small, p_big = plan(small), plan(big)
    assert p_small.kernel_names()[0] == p_big.kernel_names()[0]
    for direction, normalize in (("forward", False), ("inverse", True)):
        p_big.execute(src, dst, direction, normalize)
        gpu_device.sync()
        want = dst.copy_to_host(np.empty_like(x))[:n_small]
        p_small.execute(src, dst, direction, normalize)
        gpu_device.sync()
        got = dst.copy_to_host(np.empty_like(x))[:n_small]
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        if direction == "forward":
            shape = (-1, 1 << log_rows, 1 << log_n) if log_rows else (-1, 1 << log_n)
            head = x[:n_small].reshape(shape)[-8:]  # the last, ragged workgroup
            ref = (np.fft.fft2 if log_rows else np.fft.fft)(head.astype(np.complex128))
            assert rel_l2(got.reshape(shape)[-8:].reshape(-1), ref.reshape(-1)) <= TOL
        p_small.execute_split(re, im, o_re, o_im, direction, normalize)
        gpu_device.sync()
        for part, buf in ((want.real, o_re), (want.imag, o_im)):
            s = buf.copy_to_host(np.empty(n_big, np.float32))[:n_small]
            assert np.array_equal(s.view(np.uint32), np.ascontiguousarray(part).view(np.uint32))
    p_small.destroy()
    p_big.destroy()
