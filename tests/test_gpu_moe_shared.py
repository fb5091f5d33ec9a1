"""The f16 shared expert of long-run calls (65 rows and up): tiled matrix products instead of
the tasks that short-run calls run inside the expert launches, with the same arithmetic.

The routed experts' part of an output differs between the two paths in f32 round-off, so the
shared expert is isolated: every routed svh is zero, which makes each routed term exactly
zero, and a row's output is the shared expert's alone. It must then have the bits of a
short-run call on that row. Sizes: row tiles of 64 and 128 (from 1024 rows), hidden and
intermediate sizes whose k splits are 1, 2, 4 and 8 and whose 64-wide parts leave remainders.
"""
import numpy as np
import pytest
import torch

from exl3_amd import synth
from exl3_amd.moe import DeviceMoeLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,H,SI", [(65, 128, 128), (127, 384, 256), (128, 512, 640), (129, 1024, 128),
                                       (200, 1792, 384), (1023, 256, 512), (1024, 640, 256), (1025, 2048, 1024),
                                       (1100, 1280, 128), (1151, 384, 1152)])
def test_shared_f16_long_calls_equal_short_calls(rows, H, SI):
    cfg = synth.MoeConfig(hidden=H, inter=128, n_experts=4, top_k=2, shared_inter=SI, gate_up_K=2, down_K=2,
                          swiglu_limit=1.5)
    layer = synth.make_layer(cfg, 11 + rows, "shared")
    for lin in layer.experts:
        lin.svh = np.zeros_like(lin.svh)
    d = DeviceMoeLayer(layer, "cuda:0")
    g = torch.Generator(device="cuda:0")
    g.manual_seed(rows)
    h = torch.randn((rows, 1, H), generator=g, device="cuda:0").half()
    got = d(h).clone()
    assert got.abs().max() > 0
    odd = torch.empty(rows * H + 1, dtype=torch.float16, device="cuda:0")[1:].view(rows, 1, H)  # 2-byte aligned
    odd.copy_(h)
    assert torch.equal(d(odd), got)
    for r0 in range(0, rows, 64):
        assert torch.equal(got[r0:r0 + 64], d(h[r0:r0 + 64].contiguous())), r0
    d.close()
