"""The long-run expert kernels' part loop: one to three 128-wide k parts and more (odd and
even counts), passes of 1 to 64 rows whose last 16-row block is partly filled, every width.

Against the short-run kernels on the same rows (calls of at most 64 rows), whose sums differ
in association only: 1% of the largest output, the reference's own bound between its two
paths (glm5_gemv_nt_test.cpp:221-247)."""
import pytest
import torch

from exl3_amd import synth
from exl3_amd.moe import DeviceMoeLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,cb,H,I,rows", [(1, 0, 128, 128, 65), (2, 1, 384, 128, 66), (3, 2, 256, 384, 97),
                                           (4, 0, 640, 256, 130), (5, 1, 512, 640, 193), (6, 2, 896, 512, 66),
                                           (7, 0, 1024, 384, 79), (8, 1, 1152, 256, 321)])
def test_long_calls_match_short_calls(K, cb, H, I, rows):
    cfg = synth.MoeConfig(hidden=H, inter=I, n_experts=5, top_k=2, gate_up_K=K, gate_up_cb=cb, down_K=9 - K,
                          down_cb=(cb + 1) % 3, shared_inter=256, shared_K=4, shared_cb=cb)
    d = DeviceMoeLayer(synth.make_layer(cfg, 100 + K, "parts"), "cuda:0")
    g = torch.Generator(device="cuda:0")
    g.manual_seed(rows)
    h = torch.randn((rows, 1, H), generator=g, device="cuda:0").half()
    got = d(h).float()
    want = torch.cat([d(h[r:r + 64].contiguous()).float() for r in range(0, rows, 64)])
    assert torch.isfinite(got).all()
    assert (got - want).abs().max() <= 1e-2 * want.abs().max()
    d.close()
