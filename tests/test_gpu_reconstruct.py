"""exl3_trellis_reconstruct, bit for bit against the oracle (whose reconstruct is pinned to the
reference's): one and several 128x128 blocks, every width and codebook, a trellis base that is
4-byte aligned only, an output at an odd f16."""
import ctypes as C

import numpy as np
import pytest
import torch

import pyoracle
from exl3_amd import _lib, synth
from exl3_amd._lib import TrellisDesc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("cb", range(3))
def test_reconstruct_bits(K, cb):
    in_f, out_f = ((128, 128), (256, 128), (128, 384), (384, 256))[(K + cb) % 4]
    words = synth.trellis_words(7, f"rec{K}{cb}", in_f, out_f, K)
    su = synth.normal_f16(7, f"su{K}{cb}", (in_f,), 0.0, 1.0)
    sv = synth.normal_f16(7, f"sv{K}{cb}", (out_f,), 0.0, 1.0)
    want = pyoracle.reconstruct(words, in_f, out_f, K, cb, su, sv)
    dev = torch.device("cuda:0")
    t = torch.zeros(words.size + 2, dtype=torch.int16, device=dev)
    t[2:] = torch.from_numpy(words.reshape(-1).view(np.int16)).to(dev)
    d_su, d_sv = (torch.from_numpy(a.view(np.int16)).to(dev) for a in (su, sv))
    out = torch.zeros(in_f * out_f + 2, dtype=torch.int16, device=dev)
    desc = TrellisDesc(t.data_ptr() + 4, d_su.data_ptr(), d_sv.data_ptr(), in_f, out_f, K, cb)
    _lib.call("exl3_trellis_reconstruct", C.byref(desc), out.data_ptr() + 2, torch.cuda.current_stream().cuda_stream)
    got = out.cpu().numpy().view(np.uint16)
    assert got[0] == 0 and got[-1] == 0
    assert np.array_equal(got[1:-1].reshape(in_f, out_f), np.asarray(want).view(np.uint16).reshape(in_f, out_f))
