"""Split-layout executions whose first and last pass read and write the re and
im arrays (fg_tile_*_si / _so, fg_fft_n*_si): the bits of an in-place
interleaved execution, for every end-pass kernel, out of place and onto the
inputs, chunked, on two streams, through the allocation-free call and as a
graph."""

import numpy as np
import pytest

from conftest import normal_c64

pytestmark = pytest.mark.gpu


# (log_rows or 0, log_n, batch, chunk limit): every first and last tile, the
# narrow forms (small grids) and the tiles' own width (large ones), ragged
# last chunks, two streams; the smallest fused batches.
CASES = [
    (0, 16, 4, None), (0, 16, 131, None), (0, 16, 9, 4 << 20), (0, 17, 2, None), (0, 17, 5, 4 << 20), (0, 17, 45, None),
    (0, 18, 1, None), (0, 18, 40, None), (0, 19, 1, None), (0, 19, 19, None), (0, 20, 1, None), (0, 20, 9, None),
    (0, 20, 3, 16 << 20), (0, 21, 1, None), (0, 22, 1, None), (0, 23, 1, None),
    (4, 11, 9, None), (5, 10, 9, None), (6, 9, 9, None), (7, 8, 9, None), (7, 12, 40, None), (8, 8, 5, None),
    (8, 8, 140, 32 << 20), (9, 6, 9, None), (9, 9, 3, None), (9, 9, 40, None), (10, 5, 9, None), (10, 10, 1, None),
    (10, 10, 9, None), (10, 12, 2, None), (8, 4, 70, None), (5, 12, 3, None),
]


def _read(dev, bufs, n):
    dev.sync()
    return [b.copy_to_host(np.empty(n, np.float32)) for b in bufs]


@pytest.mark.parametrize("log_rows,log_n,batch,limit", CASES)
def test_fused_split_equals_the_in_place_execution(gpu_device, log_rows, log_n, batch, limit):
    import ferrum_gpu
    from ferrum_gpu import _native as N
    from ferrum_gpu.hip import Capture, DeviceBuffer

    saved = ferrum_gpu.fft.get_chunk_bytes()
    if limit:
        ferrum_gpu.fft.set_chunk_bytes(limit)
    try:
        plan = (ferrum_gpu.fft.Plan2D(log_rows, batch, gpu_device, log_cols=log_n) if log_rows
                else ferrum_gpu.fft.Plan1D(log_n, batch, gpu_device))
    finally:
        ferrum_gpu.fft.set_chunk_bytes(saved)
    d = plan.describe()
    n = batch << (log_rows + log_n)
    print(f"[case] log_rows={log_rows} log_n={log_n} batch={batch} {plan.kernel_names(in_place=True)[:3]} {d}", flush=True)
    fused = d["launches"] > 1 and n >= 1 << 18 and log_rows <= 10
    x = normal_c64(np.random.default_rng(1400 + log_rows + log_n), n)
    whole = DeviceBuffer(gpu_device, plan.nbytes)
    ins = [DeviceBuffer(gpu_device, 4 * n) for _ in range(2)]
    outs = [DeviceBuffer(gpu_device, 4 * n) for _ in range(2)]
    for direction, normalize in (("forward", False), ("inverse", True)):
        whole.copy_from_host(x)
        plan.execute(whole, whole, direction, normalize)
        gpu_device.sync()
        want = whole.copy_to_host(np.empty_like(x))
        parts = [np.ascontiguousarray(x.real), np.ascontiguousarray(x.imag)]
        for b, v in zip(ins, parts):
            b.copy_from_host(v)

        def same(got):
            return all(np.array_equal(g.view(np.uint32), np.ascontiguousarray(w).view(np.uint32))
                       for g, w in zip(got, (want.real, want.imag)))

        plan.execute_split(*ins, *outs, direction, normalize)
        assert same(_read(gpu_device, outs, n))
        assert all(np.array_equal(g, v) for g, v in zip(_read(gpu_device, ins, n), parts))  # inputs kept
        if 8 * n <= 64 << 20:
            for b in outs:
                b.copy_from_host(np.zeros(n, np.float32))
            plan.execute_split_noalloc(*ins, *outs, direction, normalize)
            assert same(_read(gpu_device, outs, n))
        with Capture(gpu_device, keep=[plan]) as cap:
            plan.execute_split(*ins, *outs, direction, normalize, stream=cap.stream)
        assert cap.graph.node_count == d["launches"] + (0 if fused or d["launches"] == 1 else 2)
        for _ in range(2):
            for b in outs:
                b.copy_from_host(np.zeros(n, np.float32))
            gpu_device.sync()
            cap.graph.launch()
            assert same(_read(gpu_device, outs, n))
        cap.graph.destroy()
        plan.execute_split(*ins, *ins, direction, normalize)  # onto the inputs
        assert same(_read(gpu_device, ins, n))
    assert N.last_error() == ""
    plan.destroy()


def test_fused_first_split_call_is_refused_under_capture(gpu_device):
    # as every multi-launch plan's, also where nothing needs allocating (1D)
    import ferrum_gpu
    from ferrum_gpu import _native as N
    from ferrum_gpu.hip import Capture, DeviceBuffer

    for plan in (ferrum_gpu.fft.Plan1D(18, 2, gpu_device), ferrum_gpu.fft.Plan2D(9, 2, gpu_device)):
        n = plan.batch * plan.elems
        bufs = [DeviceBuffer(gpu_device, 4 * n) for _ in range(4)]
        small = ferrum_gpu.fft.Plan1D(8, 4, gpu_device)
        buf = DeviceBuffer(gpu_device, small.nbytes)
        with Capture(gpu_device, keep=[small]) as cap:
            small.execute(buf, buf, stream=cap.stream)
            with pytest.raises(N.FerrumGpuError, match="capture"):
                plan.execute_split(*bufs, stream=cap.stream)
        cap.graph.destroy()
        small.destroy()
        plan.destroy()
