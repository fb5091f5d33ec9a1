"""The long-run expert kernels' part loop: one to three 128-wide k parts and more (odd and
even counts), passes of 1 to 64 rows whose last 16-row block is partly filled, every width.

Against the short-run kernels on the same rows (calls of at most 64 rows). Where every k range
is one slice (128, 256 or 512 wide) both add up in the same order: the same bits. Elsewhere their
sums differ in association only, so a row differs by f16 values that fell to the other side of
a rounding. A result goes through six (the projection, three in the SwiGLU, the rotation, the
weighted product and sum), each within 2^-11 of its value and 2^-11 / sqrt(3) of it on average:
were all of them drawn anew, the row's distance would be sqrt(6) sqrt(2) 2.8e-4 = 9.8e-4 of its
norm, and an element's six times that of the row's root mean square; and the reference's own
bound between its two paths holds (glm5_gemv_nt_test.cpp:221-247), 1% of the largest output."""
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
    diff, norm = (got - want)[:, 0], want[:, 0].norm(dim=1, keepdim=True)
    assert (diff.norm(dim=1, keepdim=True) <= 9.8e-4 * norm).all()
    assert (diff.abs() <= 6 * 9.8e-4 / H ** 0.5 * norm).all()
    d.close()


# one, two and four parts a k range, passes of every count of 16-row blocks, every width and
# codebook of either projection and of a shared expert
@pytest.mark.parametrize("K,cb,H,I,rows", [(1, 0, 128, 256, 65), (2, 1, 256, 128, 130), (3, 2, 512, 512, 97),
                                           (4, 1, 512, 128, 300), (4, 0, 256, 512, 66), (5, 0, 128, 512, 250),
                                           (6, 2, 512, 256, 113), (7, 1, 256, 256, 81), (8, 2, 128, 128, 700)])
def test_long_calls_equal_short_calls_in_one_slice(K, cb, H, I, rows):
    cfg = synth.MoeConfig(hidden=H, inter=I, n_experts=7, top_k=2, gate_up_K=K, gate_up_cb=cb, down_K=9 - K,
                          down_cb=(cb + 1) % 3, shared_inter=512, shared_K=K, shared_cb=(cb + 2) % 3)
    d = DeviceMoeLayer(synth.make_layer(cfg, 200 + K, "slice"), "cuda:0")
    g = torch.Generator(device="cuda:0")
    g.manual_seed(rows)
    h = torch.randn((rows, 1, H), generator=g, device="cuda:0").half()
    got = d(h).clone()
    assert torch.isfinite(got).all() and got.abs().max() > 0
    for r in range(0, rows, 64):
        assert torch.equal(got[r:r + 64], d(h[r:r + 64].contiguous())), r
    d.close()
