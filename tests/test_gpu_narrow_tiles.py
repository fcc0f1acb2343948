"""Tile passes narrowed for launches that would leave the GPU short of
workgroups (narrow_width, ferrum-gpu_amd/csrc/fft_plan.cpp): batches on both
sides of every width's limit give the bits of the same transforms in a batch
whose tiles keep their own width, and agree with the oracle."""

import numpy as np
import pytest

import oracle
from conftest import normal_c64, rel_l2

pytestmark = pytest.mark.gpu

# See test_gpu_row_tiles.py (1D twiddle recurrences and the oracle's own f32
# error); 2D plans have no recurrence and stay below it.
TOL = 5e-6


def _run(dev, plan, x, direction, normalize, in_place=False):
    from ferrum_gpu.hip import DeviceBuffer

    a = DeviceBuffer(dev, plan.nbytes)
    b = a if in_place else DeviceBuffer(dev, plan.nbytes)
    a.copy_from_host(x)
    plan.execute(a, b, direction, normalize)
    dev.sync()
    return b.copy_to_host(np.empty_like(x))


# (log_rows or 0, log_n, batches, a batch whose launches keep their own tiles):
# 1D 2^16: 8 tiles per transform, 4 columns to 4 transforms, 8 to 32, 16 to
# 128; 2^18: 32 / 16; 2^19, 2^20: 64 / 32 and 64 / 64.  2D: C / width tiles.
SHAPES = [
    (0, 16, (1, 4, 5, 32, 33, 128), 131),
    (0, 17, (1, 4, 5, 17, 39), 70),
    (0, 18, (1, 2, 3, 9, 17), 34),
    (0, 19, (1, 5), 18),
    (0, 20, (1, 2, 5), 9),
    (0, 21, (1, 2), 5),
    (0, 22, (1,), 3),
    (7, 10, (1, 8, 9, 17), 70),
    (8, 8, (1, 8, 9, 33, 65), 130),
    (9, 9, (1, 2, 3, 17), 34),
    (10, 10, (1, 2, 5), 9),
    (10, 8, (1, 4, 17), 33),
    (11, 4, (1, 64), 129),
    (12, 6, (1, 8), 17),
]


@pytest.mark.parametrize("log_rows,log_n,batches,full", SHAPES)
def test_every_width_gives_the_same_bits(gpu_device, log_rows, log_n, batches, full):
    import ferrum_gpu

    elems = 1 << (log_rows + log_n)

    def plan(batch):
        if log_rows:
            return ferrum_gpu.fft.Plan2D(log_rows, batch, gpu_device, log_cols=log_n)
        return ferrum_gpu.fft.Plan1D(log_n, batch, gpu_device)

    x = normal_c64(np.random.default_rng(1300 + log_rows + log_n), full * elems)
    for direction, normalize in (("forward", False), ("inverse", True)):
        p = plan(full)
        want = _run(gpu_device, p, x, direction, normalize)
        p.destroy()
        for i, batch in enumerate(batches):
            print(f"[case] log_rows={log_rows} log_n={log_n} batch={batch} {direction}", flush=True)
            p = plan(batch)
            got = _run(gpu_device, p, x[:batch * elems], direction, normalize)
            assert np.array_equal(got.view(np.uint32), want[:batch * elems].view(np.uint32))
            if i == 0:
                if log_rows:
                    ref = np.fft.fft2 if direction == "forward" else np.fft.ifft2
                    ref = ref(x[:batch * elems].reshape(batch, 1 << log_rows, 1 << log_n).astype(np.complex128)).reshape(-1)
                else:
                    ref = oracle.fft_1d(x[:batch * elems], log_n, direction, normalize, threads=8)
                assert rel_l2(got, ref) <= TOL
                again = _run(gpu_device, p, x[:batch * elems], direction, normalize, in_place=True)
                assert np.array_equal(again.view(np.uint32), got.view(np.uint32))
            p.destroy()
