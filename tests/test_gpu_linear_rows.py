"""exl3_trellis_linear and exl3_trellis_matmul_raw at row counts whose calls decode each
weight once for 64 or 128 rows (k_qmv_rows): tile remainders in rows and columns, odd and
even counts of its 128-wide k parts, slices of 2, 4 and 8 steps, every width and codebook.

A row's arithmetic is the slice path's, operation for operation, so the reference of every
check is the same library on the same rows 16 at a time (calls of up to 16 rows take the
slice path, which the oracle tests of test_gpu_trellis.py hold): bit for bit.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from exl3_amd import _lib, synth
from exl3_amd.trellis import (TrellisWeight, f16_from_bits, trellis_linear, trellis_linear_group,
                              trellis_linear_group_rows, trellis_matmul_raw)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def weight(dev, in_f, out_f, K, cb, seed=0):
    g = torch.Generator(device=dev)
    g.manual_seed(1000 * K + 10 * cb + in_f + out_f + seed)
    words = torch.randint(-32768, 32768, (in_f // 16, out_f // 16, 16 * K), dtype=torch.int16, generator=g, device=dev)
    su = f16_from_bits(synth.normal_f16(seed, f"suh{in_f}", (in_f,), 1.0, 0.05), dev)
    sv = f16_from_bits(synth.normal_f16(seed, f"svh{out_f}", (out_f,), 1.0, 0.05), dev)
    return TrellisWeight(words, su, sv, in_f, out_f, K, cb)


def by16(f, x):
    return torch.cat([f(x[r:r + 16]) for r in range(0, x.shape[0], 16)])


# (rows, in, out, K, codebook)
SHAPES = [
    (1023, 1024, 4096, 4, 2), (1024, 1024, 4096, 4, 1), (1025, 512, 4096, 4, 0),  # 128-row tiles
    (63, 512, 24576, 4, 1), (64, 640, 24576, 5, 0), (65, 512, 24576, 6, 2),       # 64-row tiles
    (17, 256, 33024, 3, 1), (900, 128, 8192, 7, 0), (300, 384, 20480, 8, 2),      # 1 to 3 k parts
    (2048, 128, 128, 4, 2), (1500, 896, 2176, 2, 0), (700, 768, 9344, 1, 1),
    (257, 2048, 16512, 6, 1), (129, 1152, 12416, 7, 2), (515, 1536, 6272, 5, 2),
    (515, 640, 6272, 8, 0), (515, 1280, 6272, 3, 2), (515, 640, 6400, 2, 1),
]


@pytest.mark.parametrize("rows,in_f,out_f,K,cb", SHAPES)
def test_many_rows_equal_16_row_calls(dev, rows, in_f, out_f, K, cb):
    w = weight(dev, in_f, out_f, K, cb)
    g = torch.Generator(device=dev)
    g.manual_seed(rows)
    x = torch.randn((rows, in_f), generator=g, device=dev).half()
    assert torch.equal(trellis_linear(w, x), by16(lambda v: trellis_linear(w, v), x))
    assert torch.equal(trellis_matmul_raw(w, x), by16(lambda v: trellis_matmul_raw(w, v), x))


def test_many_rows_grouped_and_special_values(dev):
    # members with their own rows and with shared ones; rows of infinities, NaN and signed
    # zeros stay in their own rows
    ws = [weight(dev, 512, 8192, 4, 1, s) for s in (1, 2, 3)]
    x = torch.randn((3, 200, 512), device=dev).half()
    x[1, 7, 3], x[1, 70, 500], x[2, 130, 0] = float("inf"), float("nan"), float("-inf")
    x[0, 20], x[0, 150] = 0.0, -0.0
    y = trellis_linear_group_rows(ws, x, 200)
    ys = trellis_linear_group(ws, x[1].contiguous())
    for m in range(3):
        for got, xm in ((y[m], x[m]), (ys[m], x[1])):
            want = by16(lambda v: trellis_linear(ws[m], v), xm.contiguous())
            assert torch.equal(got.view(torch.int16)[~want.isnan()], want.view(torch.int16)[~want.isnan()])
            assert torch.equal(got.isnan(), want.isnan())


def test_many_rows_smaller_workspace_and_unaligned_output(dev):
    # a workspace of the slice partials alone, and outputs that are only 2-byte aligned: the
    # slice path, with the same bits
    w = weight(dev, 1024, 256, 4, 2)
    rows = 2000
    x = torch.randn((rows, 1024), device=dev).half()
    want = by16(lambda v: trellis_linear(w, v), x)
    d = w.desc()
    L = _lib.lib()
    need = L.exl3_trellis_workspace_size(C.byref(d), rows, 1)
    part = 2 * rows * 256 * 4  # two k slices
    assert need >= part
    stream = torch.cuda.current_stream().cuda_stream
    for nbytes, shift in ((need, 0), (part, 0), (need, 1)):
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        y = torch.zeros(rows * 256 + 8, dtype=torch.float16, device=dev)
        _lib.call("exl3_trellis_linear", C.byref(d), x.data_ptr(), rows, y.data_ptr() + 2 * shift, ws.data_ptr(), nbytes, stream)
        assert torch.equal(y[shift:shift + rows * 256].view(rows, 256), want)
        assert not y[:shift].any() and not y[shift + rows * 256:].any()
