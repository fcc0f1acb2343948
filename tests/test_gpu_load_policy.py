"""First passes that load their input through the caches (*_loads_cached,
ferrum-gpu_amd/csrc/fft_plan.cpp): a batch below the limit gives the bits of
the same transforms at the head of a batch above it, in both layouts, and
agrees with numpy in double precision; ragged last workgroups included."""

import numpy as np
import oracle
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
CASES = [(0, n, 40, 82) for n in range(2, 13)] + [(0, 9, 20, 30), (0, 12, 30, 36)] + [(0, n, 12, 18) for n in (13, 14, 15)] + \
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


# Elements at the edges of the ranges that load through the caches (load_flags,
# ferrum-gpu_amd/csrc/pointwise_ops.cpp), ragged against the 2 and 4 elements
# per thread.
M12, M40, M80 = 12 << 17, 40 << 17, 80 << 17


@pytest.mark.parametrize("n", [M12 - 1, M12, M12 + 3, M40 - 1, M40])
@pytest.mark.parametrize("shift", [0, 1])
def test_products_by_load_policy(gpu_device, n, shift):
    """out = a * b bit for bit in both layouts and in place; shift = 1 takes
    the element-wise kernels."""
    from ferrum_gpu import pointwise
    from ferrum_gpu.hip import DeviceBuffer

    print(f"[case] products n={n} shift={shift}", flush=True)
    rng = np.random.default_rng(n + shift)
    a, b = normal_c64(rng, n), normal_c64(rng, n)
    want = oracle.cmul_interleaved(a, b)
    bufs = [DeviceBuffer(gpu_device, 8 * (n + 1)) for _ in range(3)]
    pad = np.zeros(n + 1, np.complex64)

    def put(buf, v):
        pad[shift:shift + n] = v
        buf.copy_from_host(pad)

    def get(buf):
        gpu_device.sync()
        return buf.copy_to_host(np.empty_like(pad))[shift:shift + n]

    put(bufs[0], a)
    put(bufs[1], b)
    pa, pb, po = (int(x.ptr) + 8 * shift for x in bufs)
    pointwise.cmul(gpu_device, pa, pb, po, n)
    assert np.array_equal(get(bufs[2]).view(np.uint32), want.view(np.uint32))
    pointwise.cmul(gpu_device, pa, pb, pa, n)
    assert np.array_equal(get(bufs[0]).view(np.uint32), want.view(np.uint32))
    w_re, w_im = oracle.cmul_split(a.real.copy(), a.imag.copy(), b.real.copy(), b.imag.copy())
    parts = [DeviceBuffer(gpu_device, 4 * (n + 1)) for _ in range(6)]
    fpad = np.zeros(n + 1, np.float32)
    for buf, v in zip(parts, (a.real, a.imag, b.real, b.imag)):
        fpad[shift:shift + n] = v
        buf.copy_from_host(fpad)
    pointwise.cmul_split(gpu_device, *[int(x.ptr) + 4 * shift for x in parts], n)
    gpu_device.sync()
    for buf, w in ((parts[4], w_re), (parts[5], w_im)):
        got = buf.copy_to_host(np.empty_like(fpad))[shift:shift + n]
        assert np.array_equal(got.view(np.uint32), w.view(np.uint32))


@pytest.mark.parametrize("n", [M12 - 1, M12 + 1, M80 - 1, M80])
@pytest.mark.parametrize("shift", [0, 1])
def test_conversions_by_load_policy(gpu_device, n, shift):
    from ferrum_gpu import pointwise
    from ferrum_gpu.hip import DeviceBuffer

    print(f"[case] conversions n={n} shift={shift}", flush=True)
    x = np.zeros(n + 1, np.complex64)
    x[shift:shift + n] = normal_c64(np.random.default_rng(n + 2 + shift), n)
    src, back = DeviceBuffer(gpu_device, 8 * (n + 1)), DeviceBuffer(gpu_device, 8 * (n + 1))
    re, im = DeviceBuffer(gpu_device, 4 * (n + 1)), DeviceBuffer(gpu_device, 4 * (n + 1))
    src.copy_from_host(x)
    ps, pb, pr, pi = int(src.ptr) + 8 * shift, int(back.ptr) + 8 * shift, int(re.ptr) + 4 * shift, int(im.ptr) + 4 * shift
    pointwise.deinterleave(gpu_device, ps, pr, pi, n)
    pointwise.interleave(gpu_device, pr, pi, pb, n)
    gpu_device.sync()
    for buf, part in ((re, x.real), (im, x.imag)):
        got = buf.copy_to_host(np.empty(n + 1, np.float32))[shift:shift + n]
        assert np.array_equal(got.view(np.uint32), np.ascontiguousarray(part[shift:shift + n]).view(np.uint32))
    got = back.copy_to_host(np.empty_like(x))[shift:shift + n]
    assert np.array_equal(got.view(np.uint32), x[shift:shift + n].view(np.uint32))
