"""The f16 shared expert of long-run calls (65 rows and up): as the tasks that short-run calls
run inside the expert launches, or as tiled matrix products (here from 4097 tasks on), with
the same arithmetic.

The routed experts' part of an output differs between the two paths in f32 round-off, so the
shared expert is isolated: every routed svh is zero, which makes each routed term exactly
zero, and a row's output is the shared expert's alone. It must then have the bits of a
short-run call on that row. Sizes, in either form: output tiles of 64 and of 128 (a product of
more than 512 small ones) for both products and for one, hidden and intermediate sizes whose k
splits are 1, 2, 4 and 8 and whose 64-wide parts leave remainders; 4096 tasks and the next
count that can be.
"""
import numpy as np
import pytest
import torch

from exl3_amd import synth
from exl3_amd.moe import DeviceMoeLayer

pytestmark = pytest.mark.gpu


def tasks(rows, H, SI):
    """16 rows x 16 outputs x one k split each, of the three projections."""
    def splits(n):
        return next(s for s in (8, 4, 2, 1) if n // 128 % s == 0)
    return -(-rows // 16) * (2 * (SI // 16) * splits(H) + (H // 16) * splits(SI))


TASKS = [(65, 128, 128), (127, 384, 256), (128, 512, 640), (129, 1024, 128), (200, 1792, 384),
         (1100, 256, 128), (128, 2048, 384)]
PRODUCTS = [(1023, 256, 512), (1024, 640, 256), (1025, 2048, 1024), (1100, 1280, 128), (1151, 384, 1152),
            (129, 2048, 384), (65, 4096, 512), (127, 3072, 640), (200, 1792, 1152), (600, 1152, 384),
            (1000, 640, 640), (1024, 1024, 256), (1151, 1920, 1152), (1500, 1280, 1152), (2000, 1152, 896),
            (1030, 2048, 256)]


@pytest.mark.parametrize("rows,H,SI", TASKS + PRODUCTS)
def test_shared_f16_long_calls_equal_short_calls(rows, H, SI):
    # (the 4 experts' workgroups leave room for any tasks, so the tasks' count decides)
    assert (tasks(rows, H, SI) > 4096) == ((rows, H, SI) in PRODUCTS)
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
    for shift in (1, 2, 4):  # rows that start 2-, 4- and 8-byte aligned
        at = torch.empty(rows * H + shift, dtype=torch.float16, device="cuda:0")[shift:].view(rows, 1, H)
        at.copy_(h)
        assert torch.equal(d(at), got), shift
    for r0 in range(0, rows, 64):
        assert torch.equal(got[r0:r0 + 64], d(h[r0:r0 + 64].contiguous())), r0
    # the experts' weight form changes nothing here; its workgroups have 8 waves of tasks, not 4
    d.set_tuning(weight_form=1)
    assert torch.equal(d(h), got)
    d.close()
