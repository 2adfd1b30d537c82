"""The four-elements-at-a-time decoder (`quad` in qgemv_kernels.hip) behind the
general mat-vec, the f32 precision mode and whole-matrix dequantization, at the
sizes where it can go wrong: rows of every alignment and shorter than one
quad, row counts that four does not divide, x at 4-byte addresses, groups of
several rows, ends of matrices inside a wave's range.  Values bit for bit the
oracle's; sums within GEMV_TOL (1e-4 normwise; f32 sums of at most 4100
terms in another order differ by less than 4100 * 2^-24 = 2.5e-4 of the sum of
magnitudes, measured below 1e-6)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import GEMV_TOL, normwise_err

pytestmark = pytest.mark.gpu

TYPES = ["F32", "F16", "Q4_0", "Q5_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"]


def blocks(rinf, synth, t, rows, cols, seed):
    dtype = rinf.TYPE_IDS[t]
    return dtype, synth.gen_blocks(dtype, rows, cols, seed)


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("rows,cols", [(3, 1), (5, 2), (7, 3), (9, 5), (33, 130), (6, 257), (31, 1027)])
def test_ragged_rows(rinf, synth, oracle, ctx, t, rows, cols):
    import torch
    dtype, raw = blocks(rinf, synth, t, rows, cols, rows * cols)
    x = synth.gen_x(cols, 3)
    ref = oracle.mat_vec_mul(raw, dtype, rows, cols, x)
    mat = ctx.upload(raw, dtype, rows, cols)
    buf = torch.full((cols + 16,), float("nan"), device="cuda")
    for shift in (0, 1, 3):                       # x at every 4-byte alignment, NaN around it
        d_x = buf[shift:shift + cols]
        d_x.copy_(torch.from_numpy(x))
        d_y = torch.zeros(rows, device="cuda")
        torch.cuda.synchronize()
        mat.matvec_dev(d_x, d_y)
        ctx.synchronize()
        assert normwise_err(d_y.cpu().numpy(), ref) <= GEMV_TOL
        buf.fill_(float("nan"))
    out = np.zeros(rows * cols, np.float32)
    mat.dequant_host(out)
    assert np.array_equal(out, oracle.dequantize(raw, dtype, rows * cols)[:rows * cols])
    mat.free()


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("rows,cols", [(5, 32), (12, 96), (10, 896), (3, 128), (9, 512), (17, 3840), (4099, 4096),
                                       (5000, 256)])
def test_f32_mode(rinf, synth, oracle, t, rows, cols):
    """Every shape of the kernels (units of 32 elements, a wave per row, four rows
    per workgroup), more rows than one round of workgroups, rows that start in
    the middle of a block, and the values themselves."""
    c = rinf.GpuContext(0)
    c.set_precision(rinf.PRECISION_F32)
    dtype, raw = blocks(rinf, synth, t, rows, cols, rows + cols)
    x = synth.gen_x(cols, 5)
    ref = oracle.mat_vec_mul(raw, dtype, rows, cols, x)
    y = np.zeros(rows, np.float32)
    mat = c.upload(raw, dtype, rows, cols)
    mat.matvec_host(x, y)
    assert normwise_err(y, ref) <= 1e-5
    out = np.zeros(rows * cols, np.float32)
    mat.dequant_host(out)
    assert np.array_equal(out, oracle.dequantize(raw, dtype, rows * cols)[:rows * cols])
    c.close()


@pytest.mark.parametrize("t", ["Q8_0", "Q4_K", "Q5_K", "Q6_K"])
def test_wrapped_layout(rinf, synth, oracle, ctx, t):
    """The GGUF layout of the types that an upload repacks: f32 mode and values."""
    import torch
    rows, cols = 22, 640
    dtype, raw = blocks(rinf, synth, t, rows, cols, 9)
    dev = torch.zeros(len(raw) + 512, dtype=torch.uint8, device="cuda")
    dev[:len(raw)].copy_(torch.from_numpy(raw))
    torch.cuda.synchronize()
    c = rinf.GpuContext(0)
    c.set_precision(rinf.PRECISION_F32)
    mat = c.wrap_device(dev, dtype, rows, cols)
    x = synth.gen_x(cols, 6)
    y = np.zeros(rows, np.float32)
    mat.matvec_host(x, y)
    assert normwise_err(y, oracle.mat_vec_mul(raw, dtype, rows, cols, x)) <= 1e-5
    out = np.zeros(rows * cols, np.float32)
    mat.dequant_host(out)
    assert np.array_equal(out, oracle.dequantize(raw, dtype, rows * cols)[:rows * cols])
    c.close()


def test_longest_rows(rinf, ctx):
    """A row of 2^32 - 100 columns: the step past its end does not wrap the
    counters (the loops end), and the last columns are read."""
    import torch
    cols = 2 ** 32 - 100
    nb = -(-cols // 32)
    raw = np.zeros(18 * nb, np.uint8)
    for b in (0, nb - 2, nb - 1):
        raw[18 * b:18 * b + 2] = np.array([0.5], np.float16).view(np.uint8)
        raw[18 * b + 2:18 * b + 18] = 0x99                   # every value 0.5
    mat = ctx.upload(raw, rinf.TYPE_IDS["Q4_0"], 1, cols)
    del raw
    x = torch.zeros(cols, device="cuda")
    x[0], x[40], x[cols - 1], x[cols - 5] = 1.0, 100.0, 2.0, 4.0
    y = torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    mat.matvec_dev(x, y)
    ctx.synchronize()
    assert y.item() == 3.5
    mat.free()
