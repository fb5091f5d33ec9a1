"""exl3_trellis_linear and exl3_trellis_matmul_raw at row counts whose calls decode each
weight once for 64 or 128 rows (k_qmv_rows): tile remainders in rows and columns, odd and
even counts of its 128-wide k parts, slices of 2, 4 and 8 steps, every width and codebook.

A row's arithmetic is the slice path's, operation for operation, so the reference of every
check is the same library on the same rows 16 at a time (calls of up to 16 rows take the
slice path, which the oracle tests of test_gpu_trellis.py hold): bit for bit. Every check asks
the library first which tile the call takes, so that a rule that moves cannot empty it.
"""
import ctypes as C

import pytest
import torch

from exl3_amd import _lib, synth
from exl3_amd.trellis import (TrellisWeight, f16_from_bits, trellis_linear, trellis_linear_group,
                              trellis_linear_group_rows, trellis_matmul_raw, trellis_path_info)

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


def tile(w, rows):
    """(rows, waves) of the call's tiles; at most 16 rows: the slice path."""
    info = trellis_path_info(w, rows)
    return info["rows_per_block"], info["tiles_per_workgroup"] // 8


# (rows, in, out, K, codebook)
SHAPES = [
    (1023, 1024, 4096, 4, 2), (1024, 1024, 4096, 4, 1), (1025, 512, 4096, 4, 0),  # 128-row tiles
    (63, 512, 24576, 4, 1), (64, 640, 24576, 5, 0), (65, 512, 24576, 6, 2),       # 64-row tiles
    (17, 256, 131200, 3, 1), (900, 128, 8192, 7, 0), (300, 384, 20480, 8, 2),     # 1 to 3 k parts
    (8000, 1024, 128, 4, 2), (1500, 896, 2176, 2, 0), (700, 768, 9344, 1, 1),     # one group of columns
    (257, 2048, 16512, 6, 1), (129, 1152, 12416, 7, 2), (515, 1536, 6272, 5, 2),
    (515, 640, 6272, 8, 0), (515, 1280, 6272, 3, 2), (515, 640, 6400, 2, 1),
]


@pytest.mark.parametrize("rows,in_f,out_f,K,cb", SHAPES)
def test_many_rows_equal_16_row_calls(dev, rows, in_f, out_f, K, cb):
    w = weight(dev, in_f, out_f, K, cb)
    assert tile(w, rows)[0] >= 64
    g = torch.Generator(device=dev)
    g.manual_seed(rows)
    x = torch.randn((rows, in_f), generator=g, device=dev).half()
    assert torch.equal(trellis_linear(w, x), by16(lambda v: trellis_linear(w, v), x))
    assert torch.equal(trellis_matmul_raw(w, x), by16(lambda v: trellis_matmul_raw(w, v), x))


# every width and codebook in each of the kernel's tiles, with a last row tile of 1 to 100 rows
# and columns that are no multiple of the tile's
@pytest.mark.parametrize("rows,in_f,out_f,want", [(129, 512, 8320, (64, 4)), (100, 640, 16512, (128, 4)),
                                                  (300, 384, 20608, (128, 8))])
@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("cb", range(3))
def test_every_tile_width_and_codebook(dev, rows, in_f, out_f, want, K, cb):
    w = weight(dev, in_f, out_f, K, cb, 5)
    assert tile(w, rows) == want
    x = torch.randn((rows, in_f), device=dev).half()
    assert torch.equal(trellis_linear(w, x), by16(lambda v: trellis_linear(w, v), x))


def test_many_rows_grouped_and_special_values(dev):
    # members with their own rows and with shared ones; rows of infinities, NaN and signed
    # zeros stay in their own rows
    ws = [weight(dev, 512, 8192, 4, 1, s) for s in (1, 2, 3)]
    assert tile(ws[0], 200)[0] >= 64  # one member alone; three have the more workgroups
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


def test_many_rows_smaller_workspace_and_unaligned_operands(dev):
    # rotated rows that are larger than the slice partials. The partials' workspace alone, an
    # output or an svh that starts at an odd f16 and f32 rows that start 4-byte aligned take the
    # slice path, with the same bits: it leaves the workspace past its partials as it was, where
    # the many-row path fills all of it; neither writes past it
    in_f, out_f, rows = 8192, 128, 5000
    w = weight(dev, in_f, out_f, 4, 2)
    assert tile(w, rows)[0] == 64
    x = torch.randn((rows, in_f), device=dev).half()
    want, want_raw = by16(lambda v: trellis_linear(w, v), x), by16(lambda v: trellis_matmul_raw(w, v), x)
    L = _lib.lib()
    need = L.exl3_trellis_workspace_size(C.byref(w.desc()), rows, 1)
    part = 16 * rows * out_f * 4  # 16 k slices
    assert need == rows * in_f * 2 > part
    stream = torch.cuda.current_stream().cuda_stream
    svh = torch.empty(out_f + 1, dtype=torch.float16, device=dev)
    svh[1:] = w.svh
    n = rows * out_f
    for raw, nbytes, shift, odd_svh in ((0, need, 0, 0), (0, part, 0, 0), (0, need, 1, 0), (0, need, 0, 1),
                                        (1, need, 0, 0), (1, part, 0, 0), (1, need, 1, 0), (1, need, 2, 0)):
        case = raw, nbytes, shift, odd_svh
        ws = torch.full((need + 4096,), 0xA5, dtype=torch.uint8, device=dev)
        y = torch.zeros(n + 8, dtype=torch.float32 if raw else torch.float16, device=dev)
        d = w.desc()
        if odd_svh:
            d.svh = svh.data_ptr() + 2
        _lib.call("exl3_trellis_matmul_raw" if raw else "exl3_trellis_linear", C.byref(d), x.data_ptr(), rows,
                  y.data_ptr() + y.element_size() * shift, ws.data_ptr(), nbytes, stream)
        assert torch.equal(y[shift:shift + n].view(rows, out_f), want_raw if raw else want), case
        assert not y[:shift].any() and not y[shift + n:].any(), case
        assert (ws[nbytes:] == 0xA5).all(), case
        rows_path = nbytes == need and not odd_svh and shift in ((0, 2) if raw else (0,))
        touched = int((ws[part:need] != 0xA5).sum())
        # (a byte of the rotated rows is 0xA5 by itself about once in 256)
        assert touched > (need - part) * 0.98 if rows_path else touched == 0, case
