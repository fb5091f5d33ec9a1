"""The work that is timed: calls of the EXL3 MoE layer, its MLP sub-block, the trellis
linear, the hyper-connection prepare and the tensor reconstruction, over the sizes that a
GLM-5 decode step, a speculative verify step, a batch of requests and a prefill have.

Weights are uniform random trellis words (what quantised weights look like to the decoder)
with suh of random sign near 1 and svh near 1/sqrt(in), so that projections come out at unit
scale as a model's do. Activations are N(0, 1) in f16.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "exl3-server_amd"))

CB_3INST, CB_MCG, CB_MUL1 = 0, 1, 2
NORM_EPS = 1e-5
HC_EPS = 1e-6
HC_ITERS = 20

# MoE layer shapes: hidden, intermediate, experts, top-k, gate/up K and codebook, down K and
# codebook, shared intermediate (0: none) and its K (0: f16 weights) and codebook
SMALL = dict(H=512, I=256, E=16, topk=2, gK=4, gcb=CB_MCG, dK=4, dcb=CB_MCG, SI=0, sK=0, scb=CB_MCG, scaling=1.0)
GLM5 = dict(H=4096, I=1024, E=288, topk=8, gK=4, gcb=CB_MCG, dK=5, dcb=CB_MCG, SI=1024, sK=0, scb=CB_MCG,
            scaling=2.5)
PREFILL = dict(H=4096, I=1024, E=288, topk=8, gK=4, gcb=CB_3INST, dK=5, dcb=CB_MUL1, SI=1024, sK=6, scb=CB_MCG,
               scaling=2.5)


def listed():
    return [
        # the smallest layer at one row: launches and their gaps are all of it
        dict(name="moe_small_r1", kind="moe", rows=1, same=0, hot=0, **SMALL),
        # one GLM-5 layer of a single sequence's decode step
        dict(name="moe_glm5_r1", kind="moe", rows=1, same=0, hot=0, **GLM5),
        # the same for a batch of 8 sequences: the layer's headline workload
        dict(name="moe_glm5_r8", kind="moe", rows=8, same=0, hot=0, **GLM5),
        # a batch of 64 of which 48 sequences share their token (a common prompt's start)
        dict(name="moe_glm5_r64", kind="moe", rows=64, same=48, hot=0, **GLM5),
        # a short prompt, of no round length, through the same layer
        dict(name="moe_glm5_r500", kind="moe", rows=500, same=0, hot=0, **GLM5),
        # a 2048-token prefill chunk with skewed routing (8 experts take about a quarter) and a
        # quantised shared expert, the other two codebooks in the routed experts
        dict(name="moe_prefill_r2048", kind="moe", rows=2048, same=0, hot=8, **PREFILL),
        # a decoder layer's whole MLP sub-block for a speculative verify step of 4 rows
        dict(name="block_glm5_r4", kind="block", rows=4, mult=4, **GLM5),
        # the hyper-connection prepare, with its norm, of a prefill chunk (attention has it too)
        dict(name="hc_prepare_r2048", kind="hc", rows=2048, mult=4, H=4096),
        # the qkv projection of a decode step
        dict(name="linear_qkv_r1", kind="linear", rows=1, inf=4096, outf=24576, K=4, cb=CB_MUL1),
        # the head's logits for a batch of 8
        dict(name="linear_head_r8", kind="linear", rows=8, inf=4096, outf=154880, K=6, cb=CB_MUL1),
        # the attention output projection of a prefill chunk of no round length
        dict(name="linear_o_r1000", kind="linear", rows=1000, inf=8192, outf=4096, K=4, cb=CB_MUL1),
        # one tensor to plain f16 weights when a model is loaded
        dict(name="reconstruct_4096", kind="reconstruct", inf=4096, outf=4096, K=4, cb=CB_MCG),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))


def _moe_shape(rng):
    pick = rng.random()
    if pick < 0.4:
        return dict(GLM5)
    if pick < 0.6:
        return dict(PREFILL)
    if pick < 0.7:
        return dict(SMALL)
    E = rng.choice([8, 24, 64, 160, 256])
    SI = rng.choice([0, 128 * rng.randint(1, 8)])
    return dict(H=128 * rng.randint(4, 32), I=128 * rng.randint(1, 8), E=E, topk=rng.randint(1, min(8, E)),
                gK=rng.randint(2, 6), gcb=rng.randint(0, 2), dK=rng.randint(2, 6), dcb=rng.randint(0, 2),
                SI=SI, sK=rng.choice([0, 4, 6]) if SI else 0, scb=rng.randint(0, 2), scaling=2.5)


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "block", "block", "linear", "linear", "linear", "hc", "reconstruct"])
    if kind == "moe":
        rows = _log_int(rng, 1, 1800)
        same = rows * 3 // 4 if rows >= 8 and rng.random() < 0.2 else 0
        c = _moe_shape(rng)
        return dict(kind=kind, rows=rows, same=same, hot=8 if c["E"] >= 64 and rng.random() < 0.25 else 0, **c)
    if kind == "block":
        return dict(kind=kind, rows=_log_int(rng, 1, 1200), mult=rng.choice([2, 4, 4, 4]), **_moe_shape(rng))
    if kind == "hc":
        return dict(kind=kind, rows=_log_int(rng, 1, 2048), mult=rng.choice([1, 2, 3, 4, 4, 4, 4]),
                    H=128 * _log_int(rng, 4, 32))
    if kind == "reconstruct":
        return dict(kind=kind, inf=128 * _log_int(rng, 2, 32), outf=128 * _log_int(rng, 2, 64), K=rng.randint(2, 8),
                    cb=rng.randint(0, 2))
    inf, outf = 128 * _log_int(rng, 8, 128), 128 * _log_int(rng, 4, 192)
    most = max(1, 8192 * 4096 * 1000 // (inf * outf))
    return dict(kind=kind, rows=_log_int(rng, 1, min(2048, most)), inf=inf, outf=outf, K=rng.randint(2, 8),
                cb=rng.randint(0, 2))


# --- inputs, from the seed alone ------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _normal(g, shape, std=1.0, mean=0.0, dtype=torch.float16):
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(dtype)


def _words(g, inf, outf, K):
    return torch.randint(-32768, 32768, (inf // 16, outf // 16, 16 * K), dtype=torch.int16, generator=g,
                         device="cuda")


def _scales(g, n, inf, outf):
    """suh (n, in) and svh (n, out)."""
    sign = torch.randint(0, 2, (n, inf), generator=g, device="cuda") * 2 - 1
    suh = (_normal(g, (n, inf), 0.05, 1.0, torch.float32) * sign).half()
    return suh, _normal(g, (n, outf), 0.05 / math.sqrt(inf), 1 / math.sqrt(inf))


def _linear_inputs(c, g):
    suh, svh = _scales(g, 1, c["inf"], c["outf"])
    return dict(words=_words(g, c["inf"], c["outf"], c["K"]), suh=suh[0], svh=svh[0])


def _rows(c, g):
    h = _normal(g, (c["rows"], 1, c["H"]))
    if c.get("same"):
        h[:c["same"]] = h[0]
    return h


def _moe_inputs(c, g):
    H, I, E, SI = c["H"], c["I"], c["E"], c["SI"]
    t = {}
    for j, (i, o, K) in enumerate(((H, I, c["gK"]), (H, I, c["gK"]), (I, H, c["dK"]))):
        t["words%d" % j] = [_words(g, i, o, K) for _ in range(E)]
        t["suh%d" % j], t["svh%d" % j] = _scales(g, E, i, o)
    if SI:
        for j, (i, o) in enumerate(((H, SI), (H, SI), (SI, H))):
            if c["sK"]:
                t["sh_words%d" % j] = _words(g, i, o, c["sK"])
                t["sh_suh%d" % j], t["sh_svh%d" % j] = _scales(g, 1, i, o)
            else:
                t["sh_dense%d" % j] = _normal(g, (i, o), 1 / math.sqrt(i))
    t["router"] = _normal(g, (E, H), 0.02)
    t["bias"] = _normal(g, (E,), 0.01, 0.0, torch.float32)
    if c.get("hot"):
        t["bias"][::E // c["hot"]][:c["hot"]] += 0.23  # a quarter of the selections
    return t


def _hc_inputs(c, g):
    N, H = c["mult"], c["H"]
    W = (2 + N) * N
    return dict(fn=_normal(g, (W, N * H), 1 / math.sqrt(N * H), 0.0, torch.float32),
                base=_normal(g, (W,), 0.5, 0.0, torch.float32),
                scale=torch.tensor([1.3, 0.7, 2.1], device="cuda"),
                norm_w=_normal(g, (H,), 0.2, 1.0),
                streams=_normal(g, (c["rows"], N, H)))


def _inputs(c, seed):
    g = _gen(seed)
    if c["kind"] in ("linear", "reconstruct"):
        t = _linear_inputs(c, g)
        if c["kind"] == "linear":
            t["x"] = _normal(g, (c["rows"], c["inf"]))
        return t
    if c["kind"] == "hc":
        return _hc_inputs(c, g)
    t = _moe_inputs(c, g)
    t.update(_hc_inputs(c, g) if c["kind"] == "block" else dict(h=_rows(c, g)))
    return t


def _bits(t):
    return t.cpu().numpy().view(np.uint16)


def _layer(c, t):
    from exl3_amd import synth
    from exl3_amd.moe import DeviceMoeLayer
    H, I, SI = c["H"], c["I"], c["SI"]
    cfg = synth.MoeConfig(hidden=H, inter=I, n_experts=c["E"], top_k=c["topk"], routed_scaling_factor=c["scaling"],
                          swiglu_limit=10.0, shared_inter=SI, gate_up_K=c["gK"], gate_up_cb=c["gcb"],
                          down_K=c["dK"], down_cb=c["dcb"], shared_K=c["sK"], shared_cb=c["scb"])
    shapes = ((H, I, c["gK"], c["gcb"]), (H, I, c["gK"], c["gcb"]), (I, H, c["dK"], c["dcb"]))
    suh, svh = [_bits(t["suh%d" % j]) for j in range(3)], [_bits(t["svh%d" % j]) for j in range(3)]
    experts, words = [], {}
    for e in range(c["E"]):
        for j, (i, o, K, cb) in enumerate(shapes):
            experts.append(synth.Linear(i, o, suh=suh[j][e], svh=svh[j][e], K=K, cb=cb))
            words[3 * e + j] = t["words%d" % j][e]
    shared = None
    if SI:
        shared = []
        for j, (i, o) in enumerate(((H, SI), (H, SI), (SI, H))):
            if c["sK"]:
                shared.append(synth.Linear(i, o, suh=_bits(t["sh_suh%d" % j][0]), svh=_bits(t["sh_svh%d" % j][0]),
                                           K=c["sK"], cb=c["scb"]))
                words[("shared", j)] = t["sh_words%d" % j]
            else:
                shared.append(synth.Linear(i, o, dense=_bits(t["sh_dense%d" % j])))
    layer = synth.MoeLayer(cfg, experts, shared, _bits(t["router"]), t["bias"].cpu().numpy())
    return DeviceMoeLayer(layer, "cuda:0", words=words)


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "moe":
        return kind, _layer(case, t), t["h"]
    if kind in ("block", "hc"):
        from exl3_amd.hc import DeviceHcSite
        site = DeviceHcSite(case["mult"], HC_ITERS, HC_EPS, t["fn"], t["base"], t["scale"])
        layer = _layer(case, t) if kind == "block" else None
        return kind, layer, site, t["norm_w"], t["streams"]
    from exl3_amd.trellis import TrellisWeight
    w = TrellisWeight(t["words"], t["suh"], t["svh"], case["inf"], case["outf"], case["K"], case["cb"])
    return kind, w, t.get("x")


def run(state):
    kind = state[0]
    if kind == "moe":
        _, layer, h = state
        return layer(h)
    if kind == "block":
        from exl3_amd.hc import moe_block
        _, layer, site, norm_w, streams = state
        return moe_block(layer, site, norm_w, NORM_EPS, streams)
    if kind == "hc":
        from exl3_amd.hc import hc_prepare
        _, _, site, norm_w, streams = state
        return hc_prepare(streams, site, norm_w, NORM_EPS)
    from exl3_amd.trellis import trellis_linear, trellis_reconstruct
    _, w, x = state
    return trellis_linear(w, x) if kind == "linear" else trellis_reconstruct(w)


# --- what a pass cannot do without ----------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    if kind in ("linear", "reconstruct"):
        n = c["inf"] * c["outf"]
        b = n * c["K"] / 8 + 2 * (c["inf"] + c["outf"])
        if kind == "reconstruct":
            return dict(bytes=b + 2 * n, flops=2 * 7 * n)
        return dict(bytes=b + 2 * c["rows"] * (c["inf"] + c["outf"]), flops=2 * c["rows"] * n)
    r, H = c["rows"], c["H"]
    b = f = 0.0
    if kind != "moe":
        N = c["mult"]
        W = (2 + N) * N
        b += 4 * W * N * H + 2 * r * H * N + 4 * r * (N + N * N)
        f += 2 * r * N * H * (W + 2)
        if kind == "hc":
            return dict(bytes=b + 2 * r * H, flops=f)
        b += 2 * r * H * N  # the new streams
        f += 2 * r * H * N * (N + 1)
    I, E, k, SI = c["I"], c["E"], c["topk"], c["SI"]
    distinct = E * (1 - (1 - k / E) ** max(1, r - max(0, c.get("same", 0) - 1)))
    b += distinct * (2 * H * I * c["gK"] + I * H * c["dK"]) / 8 + 2 * E * H
    b += 3 * H * SI * (c["sK"] or 16) / 8
    f += 2.0 * r * (3 * H * (k * I + SI) + H * E)
    if kind == "moe":
        b += 4 * r * H
    return dict(bytes=b, flops=f)


def tolerance(case):
    """About four times the distance from exact() (f16 roundings of the rotated inputs, the
    projections and the results): 3.6e-4 for a linear and a prepare, 7.5e-4 to 9.4e-4 for a
    layer. In the sub-block a last-bit change of the normed rows can tip a near-tie of the
    routing, which swaps one of a row's experts: 1.7e-2 was seen against exact() over 1173
    rows. The reconstruction is defined to the bit."""
    return {"reconstruct": "exact", "linear": {"rel": 1.5e-3}, "hc": {"rel": 1.5e-3}, "moe": {"rel": 3e-3},
            "block": {"rel": 2e-2}}[case["kind"]]


# --- the same results in 64 bits --------------------------------------------------------

_TABLES = {}


def _codebook(cb):
    """The 65,536 weights of a codebook as f64 (each an f16 value)."""
    if cb not in _TABLES:
        s = np.arange(65536, dtype=np.uint64)
        if cb == CB_MUL1:
            h = (s * np.uint64(0x83DCD12D)) & np.uint64(0xFFFFFFFF)
            total = sum((h >> np.uint64(8 * i)) & np.uint64(255) for i in range(4))
            v = (np.uint64(0x6400) + total).astype(np.uint16).view(np.float16).astype(np.float64)
            a, b = np.array([0x1EEE, 0xC931], np.uint16).view(np.float16).astype(np.float64)
            w = (v * a + b).astype(np.float16)
        else:
            m, add = ((89226354, 64248484), (0xCBAC1FED, 0))[cb]
            h = (s * np.uint64(m) + np.uint64(add)) & np.uint64(0xFFFFFFFF)
            h = ((h & np.uint64(0x8FFF8FFF)) ^ np.uint64(0x3B603B60)).astype(np.uint32)
            halves = h.view(np.uint16).view(np.float16).astype(np.float64).reshape(-1, 2)
            w = (halves[:, 0] + halves[:, 1]).astype(np.float16)
        p = np.arange(256)
        lane, i = p >> 3, p & 7
        q = i & 3
        element = (2 * (lane & 3) + np.where(q < 2, q, q + 6)) * 16 + (lane >> 2) + 8 * (i >> 2)
        _TABLES[cb] = torch.from_numpy(w.astype(np.float64)).cuda(), torch.from_numpy(np.argsort(element)).cuda()
    return _TABLES[cb]


def _decode(words, K, cb):
    """(k tiles, n tiles, 16 K) int16 -> the rotated-basis weights (in, out) in f64."""
    table, at = _codebook(cb)
    w = words.view(torch.int32).long() & 0xFFFFFFFF
    last = (at + 1) * K - 1  # the last ring bit of each element's state
    shift = 31 - (last & 31)
    lo, hi = w[..., (last >> 5) % (8 * K)], w[..., ((last >> 5) - 1) % (8 * K)] & 0xFFFF
    tile = table[((lo >> shift) | (hi << (32 - shift))) & 0xFFFF]
    kt, nt = words.shape[:2]
    return tile.view(kt, nt, 16, 16).permute(0, 2, 1, 3).reshape(16 * kt, 16 * nt)


def _hadamard(x):
    """The orthonormal 128-point transform of every 128 values of the last axis."""
    if "H" not in _TABLES:
        h = torch.ones((1, 1), dtype=torch.float64)
        while h.shape[0] < 128:
            h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
        _TABLES["H"] = (h / math.sqrt(128)).cuda()
    return (x.reshape(-1, 128) @ _TABLES["H"]).view(x.shape)


def _exact_linear(x, words, suh, svh, K, cb):
    xh = _hadamard(x * suh.double())
    step = max(1, (1 << 25) // (256 * words.shape[1]))
    y = 0
    for k in range(0, words.shape[0], step):
        y = y + xh[:, 16 * k:16 * (k + step)] @ _decode(words[k:k + step], K, cb)
    return _hadamard(y) * svh.double()


def _swiglu(g, u):
    g = g.clamp(max=10.0)
    return g * torch.sigmoid(g) * u.clamp(-10.0, 10.0)


def _exact_moe(c, t, h):
    score = torch.sigmoid(h @ t["router"].double().T)
    ids = (score + t["bias"].double()).topk(c["topk"], dim=-1).indices
    w = score.gather(1, ids)
    w = w / (w.sum(-1, keepdim=True) + 1e-20) * c["scaling"]
    out = torch.zeros_like(h)
    for e in torch.unique(ids).tolist():
        row, rank = (ids == e).nonzero(as_tuple=True)
        lin = lambda x, j: _exact_linear(  # noqa: E731
            x, t["words%d" % j][e], t["suh%d" % j][e], t["svh%d" % j][e], c["dK" if j == 2 else "gK"],
            c["dcb" if j == 2 else "gcb"])
        y = lin(_swiglu(lin(h[row], 0), lin(h[row], 1)), 2)
        out.index_add_(0, row, y * w[row, rank, None])
    if c["SI"]:
        if c["sK"]:
            lin = lambda x, j: _exact_linear(  # noqa: E731
                x, t["sh_words%d" % j], t["sh_suh%d" % j][0], t["sh_svh%d" % j][0], c["sK"], c["scb"])
        else:
            lin = lambda x, j: x @ t["sh_dense%d" % j].double()  # noqa: E731
        out = out + lin(_swiglu(lin(h, 0), lin(h, 1)), 2)
    return out


def _exact_hc(c, t):
    N, s = c["mult"], t["streams"].double()
    x = s.flatten(1)
    v = (x @ t["fn"].double().T) / torch.sqrt(x.square().mean(-1, keepdim=True) + HC_EPS)
    base, scale = t["base"].double(), t["scale"].double()
    pre = torch.sigmoid(v[:, :N] * scale[0] + base[:N]) + HC_EPS
    post = 2 * torch.sigmoid(v[:, N:2 * N] * scale[1] + base[N:2 * N])
    comb = torch.softmax((v[:, 2 * N:] * scale[2] + base[2 * N:]).view(-1, N, N), -1) + HC_EPS
    comb = comb / (comb.sum(-2, keepdim=True) + HC_EPS)
    for _ in range(HC_ITERS - 1):
        comb = comb / (comb.sum(-1, keepdim=True) + HC_EPS)
        comb = comb / (comb.sum(-2, keepdim=True) + HC_EPS)
    y = (pre[:, :, None] * s).sum(1)
    y = y / torch.sqrt(y.square().mean(-1, keepdim=True) + NORM_EPS) * t["norm_w"].double()
    return y, post, comb


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    if c["kind"] == "linear":
        return _exact_linear(t["x"].double(), t["words"], t["suh"], t["svh"], c["K"], c["cb"])
    if c["kind"] == "reconstruct":
        w = _hadamard(_decode(t["words"], c["K"], c["cb"]).T.contiguous()).T * t["suh"].double()[:, None]
        return _hadamard(w.contiguous()) * t["svh"].double()
    if c["kind"] == "moe":
        return _exact_moe(c, t, t["h"].view(c["rows"], -1).double()).view(t["h"].shape)
    y, post, comb = _exact_hc(c, t)
    if c["kind"] == "hc":
        return y, post, comb
    out = _exact_moe(c, t, y)
    return post[:, :, None] * out[:, None, :] + comb.transpose(1, 2) @ t["streams"].double()
