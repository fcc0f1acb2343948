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
# on 256 CUs both sides of every width's limit (narrow_width; each limit is
# asked of the rule itself in test_plan_rules.py).  Transforms or images up to
# which a launch takes 4 / 8 / 16 columns: 2^16 4 / 32 / 64; 2^17 first pass 2 /
# 16 / 32, last 4; 2^18 first 1 / 8 / 16, last 4 / 16; 2^19 first 1 / 8, last 2 / 8;
# 2^20 1 / 4; 2^21, 2^22 - / - / 1; 128 rows x 1024 - / 8 / 16; 256 x 256 4 / 32 /
# 64; 512 x 512 2 / 16; 1024 x 1024 1 / 4; 1024 x 256 4 / 16; 2048 x 16 64; 4096 x
# 64 16.
SHAPES = [
    (0, 16, (1, 4, 5, 32, 33, 64, 65), 131),
    (0, 17, (1, 2, 3, 4, 5, 16, 17, 32, 33), 70),
    (0, 18, (1, 2, 4, 5, 8, 9, 16, 17), 34),
    (0, 19, (1, 2, 3, 8, 9), 18),
    (0, 20, (1, 2, 4, 5), 9),
    (0, 21, (1, 2), 5),
    (0, 22, (1, 2), 3),
    (7, 10, (1, 8, 9, 16, 17), 70),
    (8, 8, (1, 4, 5, 32, 33, 64, 65), 130),
    (9, 9, (1, 2, 3, 16, 17), 34),
    (10, 10, (1, 2, 4, 5), 9),
    (10, 8, (1, 4, 5, 16, 17), 33),
    (11, 4, (1, 64, 65), 129),
    (12, 6, (1, 16, 17), 33),
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
