"""exl3_trellis_linear, its grouped form and exl3_trellis_matmul_raw at widths where a
workgroup of k_qmv takes 2 or 4 column blocks: last groups of 1 to 3 blocks, slices of 2, 4
and 8 steps, every width and codebook, members of one launch.

An output's operations and their order do not depend on the group, so the reference is the
same columns in calls too narrow for groups (held by the oracle tests of
test_gpu_trellis.py): bit for bit.
"""
import pytest
import torch

from exl3_amd import synth
from exl3_amd.trellis import TrellisWeight, f16_from_bits, trellis_linear, trellis_linear_group, trellis_matmul_raw

pytestmark = pytest.mark.gpu


def tensors(in_f, out_f, K, seed=0):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(100 * K + in_f + out_f + seed)
    words = torch.randint(-32768, 32768, (in_f // 16, out_f // 16, 16 * K), dtype=torch.int16, generator=g,
                          device="cuda:0")
    su = f16_from_bits(synth.normal_f16(seed, f"suh{in_f}", (in_f,), 1.0, 0.05), "cuda:0")
    sv = f16_from_bits(synth.normal_f16(seed, f"svh{out_f}", (out_f,), 1.0, 0.05), "cuda:0")
    return words, su, sv


# (rows, in, out, K, codebook)
SHAPES = [
    (9, 4096, 192 * 128, 4, 2), (16, 896, 221 * 128, 3, 0), (16, 1280, 309 * 128, 6, 1),   # 2 blocks, the last 2, 1, 1
    (8, 1152, 345 * 128, 5, 2), (16, 128, 3073 * 128, 4, 1),                               # 2, the last alone
    (15, 2048, 768 * 128, 7, 2), (2, 1024, 5001 * 128, 1, 1),                              # 4, the last 4, 1
    (4, 1152, 970 * 128, 8, 0), (3, 256, 8191 * 128, 2, 0),                                # 4, the last 2, 3
]


@pytest.mark.parametrize("rows,in_f,out_f,K,cb", SHAPES)
def test_groups_equal_narrow_calls(rows, in_f, out_f, K, cb):
    words, su, sv = tensors(in_f, out_f, K)
    g = torch.Generator(device="cuda:0")
    g.manual_seed(rows)
    x = torch.randn((rows, in_f), generator=g, device="cuda:0").half()
    w = TrellisWeight(words, su, sv, in_f, out_f, K, cb)
    y, raw = trellis_linear(w, x), trellis_matmul_raw(w, x)
    step = 64 * 128
    for c in range(0, out_f, step):
        n = min(step, out_f - c)
        part = TrellisWeight(words[:, c // 16:(c + n) // 16].contiguous(), su, sv[c:c + n].clone(), in_f, n, K, cb)
        assert torch.equal(trellis_linear(part, x), y[:, c:c + n]), c
        assert torch.equal(trellis_matmul_raw(part, x), raw[:, c:c + n]), c


def test_groups_of_members():
    # three members of 9 x 59 workgroups each: groups of 2 in the joint launch, none alone
    in_f, out_f, K, cb = 1152, 59 * 128, 4, 1
    ws = [TrellisWeight(*tensors(in_f, out_f, K, s), in_f, out_f, K, cb) for s in (1, 2, 3)]
    x = torch.randn((16, in_f), device="cuda:0").half()
    y = trellis_linear_group(ws, x)
    for m in range(3):
        assert torch.equal(y[m], trellis_linear(ws[m], x))
