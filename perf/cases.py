"""What this framework is measured on: the calls a user of the expert layer
makes, over the range of sizes they are made at.

Kinds of case:
  layer     SimpleMoE forward without autograd (serving): decode steps of one
            to a few hundred tokens, prefill chunks, whole prompts
  train     one training step of the layer after an optimizer update: the fp8
            weights are refreshed, then forward and backward under autograd
  experts   the expert FFN alone on rows that are already dispatched (one
            rank's share behind a caller's own dispatcher), skewed loads
  gemm      the grouped GEMM alone, on plain [E, N, K] weights
  dispatch  expert sort + permute + 1x128 quantisation of a batch

Shapes are the benchmark's and the tests' own: the tiny layer (H 1024, I 2048,
E 8, top-2), Mixtral (4096, 14336, 8, 2), Qwen3-30B-A3B (2048, 768, 128, 8),
DeepSeek-V3's local share (7168, 2048, 32 experts, top-8) and GPT-OSS (2880,
2880, 32, 4: not multiples of 128); drawn cases take generic sizes as well.
"""
import os
import sys

import torch

_PKG = os.path.abspath("system-lab_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

SHAPES = {
    "tiny": dict(H=1024, I=2048, E=8, K=2),
    "mixtral": dict(H=4096, I=14336, E=8, K=2),
    "qwen3": dict(H=2048, I=768, E=128, K=8),
    "dsv3": dict(H=7168, I=2048, E=32, K=8),
    "gptoss": dict(H=2880, I=2880, E=32, K=4),
}
MAX_FLOPS = 5.8e12   # the largest listed case (Mixtral, 8192 tokens)


def _case(kind, T, recipe="blockwise", gate=False, shape=None, **dims):
    c = dict(kind=kind, T=T, recipe=recipe, gate=gate)
    c.update(SHAPES[shape] if shape else {})
    c.update(dims)
    return c


def listed():
    return [
        # one token of a single decoding stream: 8 of 128 experts, launch- and weight-bound
        dict(name="decode_1_qwen3", **_case("layer", 1, gate=True, shape="qwen3")),
        # a decode batch of 32 streams on few, large experts
        dict(name="decode_32_mixtral", **_case("layer", 32, gate=True, shape="mixtral")),
        # a decode batch of 128 streams: every expert has a few rows
        dict(name="decode_128_qwen3", **_case("layer", 128, gate=True, shape="qwen3")),
        # a chunk of a prompt, ragged: about 60 rows an expert
        dict(name="prefill_1000_qwen3", **_case("layer", 1000, shape="qwen3")),
        # a ragged chunk on dimensions that are not multiples of 128, E8M0 scales
        dict(name="prefill_777_gptoss_e8m0", **_case("layer", 777, recipe="e8m0", shape="gptoss")),
        # whole prompts: the benchmark's Mixtral layer forward
        dict(name="prefill_8192_mixtral", **_case("layer", 8192, shape="mixtral")),
        # a training step of a small layer
        dict(name="train_2048_tiny", **_case("train", 2048, shape="tiny")),
        # the benchmark's forward + backward at Qwen3's shape
        dict(name="train_16384_qwen3", **_case("train", 16384, shape="qwen3")),
        # a training step at GPT-OSS's dimensions, E8M0 scales
        dict(name="train_4096_gptoss_e8m0", **_case("train", 4096, recipe="e8m0", shape="gptoss")),
        # the benchmark's DeepSeek-V3 local experts, 65536 rows under Zipf loads
        dict(name="experts_65536_dsv3", **_case("experts", 8192, shape="dsv3")),
        # a grouped GEMM call of 8192 rows over 32 experts, plain weights
        dict(name="gemm_8192_plain", **_case("gemm", 1024, shape=None, H=7168, I=2048, E=32, K=8)),
        # the benchmark's permute + quantise batch
        dict(name="dispatch_16384", **_case("dispatch", 16384, shape=None, H=7168, I=0, E=256, K=8)),
    ]


def draw(rng):
    kind = rng.choice(["layer"] * 6 + ["train"] * 3 + ["experts", "gemm", "dispatch"])
    recipe = rng.choice(["blockwise", "blockwise", "e8m0"])
    if rng.random() < 0.6:
        dims = dict(SHAPES[rng.choice(sorted(SHAPES))])
    else:  # generic widths, multiples of 16, and expert counts
        E = rng.choice([8, 16, 24, 32, 60, 64, 96, 128])
        dims = dict(H=16 * int(2 ** rng.uniform(6, 8.5)), I=16 * int(2 ** rng.uniform(5, 7.5)), E=E,
                    K=rng.randint(1, min(8, E)))
    if kind in ("experts", "gemm"):  # whole 128-wide blocks
        dims["H"], dims["I"] = -(-dims["H"] // 128) * 128, -(-dims["I"] // 128) * 128
    lo = {"layer": 0, "train": 8, "experts": 4, "gemm": 4, "dispatch": 2}[kind]
    T = int(2 ** rng.uniform(lo, 14))
    gate = kind == "layer" and T <= 512 and rng.random() < 0.7
    c = dict(kind=kind, T=T, recipe="blockwise" if kind in ("gemm", "dispatch") else recipe, gate=gate, **dims)
    while work(c)["flops"] > MAX_FLOPS:
        c["T"] = c["T"] * 2 // 3
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 * seed + salt)
    return g


def _randn(shape, seed, salt, std=1.0):
    return torch.randn(shape, generator=_gen(seed, salt), device="cuda", dtype=torch.float32) * std


def _bf16(shape, seed, salt, std=1.0):
    return _randn(shape, seed, salt, std).to(torch.bfloat16)


def _weights(shape, seed, salt, std):
    """bf16 [E, N, K] ~ N(0, std), an expert at a time."""
    g = _gen(seed, salt)
    w = torch.empty(shape, device="cuda", dtype=torch.bfloat16)
    for e in range(shape[0]):
        w[e] = torch.randn(shape[1:], generator=g, device="cuda") * std
    return w


def _zipf_offsets(R, E, seed):
    """Row offsets of Zipf(1.2) loads, an eighth of the experts empty, the
    ranks dealt to the experts at random."""
    live = max(1, E - E // 8)
    share = torch.arange(1, live + 1, dtype=torch.float64).pow(-1.2)
    n = torch.zeros(E, dtype=torch.int64)
    n[:live] = (share / share.sum() * R).floor().long()
    n[0] += R - int(n.sum())
    n = n[torch.randperm(E, generator=torch.Generator().manual_seed(seed))]
    off = torch.zeros(E + 1, dtype=torch.int32)
    off[1:] = n.cumsum(0).int()
    return off.cuda()


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    T, H, I, E, K = (case[k] for k in ("T", "H", "I", "E", "K"))
    kind = case["kind"]
    d = {}
    if kind == "dispatch":
        x = _randn((T, H), seed, 1)
        x = torch.where(torch.rand((T, H), generator=_gen(seed, 8), device="cuda") < 1e-3, x * 50, x)
        d["x"] = x.to(torch.bfloat16)
        lg = _randn((T, E), seed, 2) + _randn((E,), seed, 3, 0.5)
        d["idx"] = lg.topk(K, dim=1).indices.int().contiguous()
        return d
    if kind in ("experts", "gemm"):
        d["x"] = _bf16((T * K, H), seed, 1)
        d["offsets"] = _zipf_offsets(T * K, E, seed)
        if kind == "gemm":
            d["w"] = _weights((E, I, H), seed, 4, 0.02)
            return d
    else:
        d["x"] = _bf16((T, H), seed, 1)
        if case["gate"]:
            d["w_gate"] = _randn((H, E), seed, 2, H ** -0.5)
        else:
            d["logits"] = _randn((T, E), seed, 2)
        if kind == "train":
            d["dout"] = _bf16((T, H), seed, 6, 1e-3)
    d["w1"] = _weights((E, 2 * I, H), seed, 4, 0.02)
    d["w2"] = _weights((E, H, I), seed, 5, 0.02)
    return d


def prepare(case, seed):
    import smoe
    d = _inputs(case, seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind == "dispatch":
        s.update(x=d["x"], idx=d["idx"])
    elif kind in ("experts", "gemm"):
        scale = "pow2" if case["recipe"] == "e8m0" else "amax"
        rows = torch.arange(d["x"].shape[0], dtype=torch.int32, device="cuda")
        s["xq"], s["xs"] = smoe.permute_quant_rows(d["x"], rows, 1, scale=scale)
        s["offsets"] = d["offsets"]
        if kind == "gemm":
            s["w"], s["ws"] = smoe.quantize_weight_blockwise(d["w"])
        else:
            form = smoe.ops.packed_e8m0_ok if scale == "pow2" else smoe.packed_gemm_ok
            for n in ("w1", "w2"):
                wq, s[n + "s"] = smoe.quantize_weight_blockwise(d[n], scale=scale)
                s[n] = smoe.pack_weight_fp8(wq) if form(wq.shape[1], wq.shape[2]) else wq
    else:
        m = smoe.SimpleMoE(case["H"], case["I"], case["E"], case["K"], device="cuda", recipe=case["recipe"])
        with torch.no_grad():
            m.w1.data, m.w2.data = d["w1"], d["w2"]
            m.w_gate.copy_(d["w_gate"] if case["gate"] else torch.zeros_like(m.w_gate))
        s.update(m=m, x=d["x"], logits=d.get("logits"))
        if kind == "train":
            s["x"].requires_grad_(True)
            s["logits"].requires_grad_(True)
            s["dout"] = d["dout"]
        else:
            m.gemm_weights()  # a server has its fp8 weights before the first request
    return s


def run(s):
    import smoe
    case = s["case"]
    kind = case["kind"]
    if kind == "dispatch":
        xq, *rest = smoe.permute_quant(s["x"], s["idx"], case["E"])
        return [xq.view(torch.uint8), *rest]
    if kind == "gemm":
        return smoe.grouped_gemm_fp8(s["xq"], s["xs"], s["w"], s["ws"], s["offsets"])
    if kind == "experts":
        e8 = case["recipe"] == "e8m0"
        hq, hs = smoe.grouped_gemm_fp8_swiglu(s["xq"], s["xs"], s["w1"], s["w1s"], s["offsets"],
                                              scale="pow2" if e8 else "amax")
        return smoe.grouped_gemm_fp8(hq, hs, s["w2"], s["w2s"], s["offsets"], e8m0=e8)
    m = s["m"]
    if kind == "layer":
        with torch.no_grad():
            return m(s["x"], s["logits"])
    for t in (s["x"], s["logits"], m.w1, m.w2):
        t.grad = None
    m.refresh_fp8_cache()  # the optimizer has just written the weights
    out = m(s["x"], s["logits"])
    out.backward(s["dout"])
    return [out.detach(), s["x"].grad, s["logits"].grad, m.w1.grad, m.w2.grad]


# ------------------------------------------------------------------- work
def work(case):
    T, H, I, E, K = (case[k] for k in ("T", "H", "I", "E", "K"))
    R, kind = T * K, case["kind"]
    if kind == "dispatch":
        G = -(-H // 128)
        return {"bytes": T * H * 2 + R * H + R * G * 4 + R * 4 + R * 8 + (E + 1) * 4, "flops": 2 * T * H}
    live = E * (1 - (1 - K / E) ** T)  # experts that get a row
    if kind in ("experts", "gemm"):
        live = min(E - E // 8, R)
        n = I if kind == "gemm" else 3 * I
        out = I if kind == "gemm" else H
        return {"bytes": int(R * H * (1 + 4 / 128) + live * n * H + R * out * 2), "flops": 2 * R * n * H}
    if kind == "layer":
        gate = H * E * 4 if case["gate"] else T * E * 4
        return {"bytes": int(2 * T * H * 2 + gate + live * 3 * I * H), "flops": 6 * R * I * H}
    # train: bf16 weights in, bf16 gradients out, fp8 weights once forward and once backward
    return {"bytes": int(E * 3 * I * H * 2 * 2 + live * 3 * I * H * 2 + 4 * T * H * 2 + 2 * T * E * 4),
            "flops": 18 * R * I * H}


def tolerance(case):
    """A bf16 result rounds to 2^-9 of a value; two correct orders of the fp32
    sums round a few values in a thousand apart.  Behind a requantisation such
    a step can move an fp8 value by one step of 1/16 to 1/8."""
    return {"dispatch": "exact", "gemm": {"rel": 2e-3, "max": 0.02}, "experts": {"rel": 6e-3, "max": 0.1},
            "layer": {"rel": 8e-3, "max": 0.15}, "train": {"rel": 1e-2, "max": 0.4}}[case["kind"]]


# ------------------------------------------------------- 64-bit statement
def _fake(v, pow2):
    """v [..., D] in groups of 128 along the last dimension (the last one
    zero-padded): scale amax/448, or the least power of two at or above it;
    round to e4m3; the dequantised values in 64 bits."""
    D = v.shape[-1]
    pad = -D % 128
    f = torch.nn.functional.pad(v.float(), (0, pad)).unflatten(-1, (-1, 128))
    return _e4m3(f, f.abs().amax(-1, keepdim=True), pow2).flatten(-2)[..., :D]


def _e4m3(f, amax, pow2):
    s = (amax.double() / 448).float()  # RN(amax/448): a scalar divisor may become a multiplication
    if pow2:
        m, e = torch.frexp(s)
        s = torch.where(m == 0.5, s, torch.ldexp(torch.ones_like(s), e))
    s = torch.where(amax == 0, torch.ones_like(s), s)
    q = (f.double() / s.double()).float()
    return q.clamp(-448, 448).to(torch.float8_e4m3fn).double() * s.double()


def _fake_cols(v, pow2):
    return _fake(v.t(), pow2).t()


def _fake_weight(w, pow2):
    """128x128 blocks of w [N, K]."""
    N, K = w.shape
    f = torch.nn.functional.pad(w.float(), (0, -K % 128, 0, -N % 128))
    f = f.unflatten(0, (-1, 128)).unflatten(2, (-1, 128))
    q = _e4m3(f, f.abs().amax((1, 3), keepdim=True), pow2)
    return q.flatten(2, 3).flatten(0, 1)[:N, :K]


def _b(v):
    """Rounded to bf16, as the tensors between two stages are."""
    return v.to(torch.bfloat16).double()


def _ffn(xe, w1, w2, pow2):
    c1 = _b(xe @ w1.t())
    g, u = c1.chunk(2, dim=1)
    h = torch.nn.functional.silu(g) * u
    return g, u, h, _b(_fake(h, pow2) @ w2.t())


def exact(case, seed):
    d = _inputs(case, seed)
    T, E, K, kind = case["T"], case["E"], case["K"], case["kind"]
    p2 = case["recipe"] == "e8m0"
    if kind == "dispatch":
        return None
    x = _fake(d["x"], p2)
    if kind in ("experts", "gemm"):
        off = d["offsets"].tolist()
        out = []
        for e in range(E):
            rows = x[off[e]:off[e + 1]]
            if kind == "gemm":
                out.append(rows @ _fake_weight(d["w"][e], p2).t())
            else:
                w1, w2 = _fake_weight(d["w1"][e], p2), _fake_weight(d["w2"][e], p2)
                out.append(_ffn(rows, w1, w2, p2)[3])
        return torch.cat(out)
    logits = d["x"].double() @ d["w_gate"].double() if case["gate"] else d["logits"].double()
    p = logits.softmax(1)
    pk, idx = p.topk(K, dim=1)
    wk = pk / pk.sum(1, keepdim=True)
    flat, wf = idx.flatten(), wk.flatten()
    out = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    if kind == "train":
        dout = d["dout"].double()
        dx = torch.zeros_like(out)
        dw = torch.zeros_like(wf)
        dw1 = torch.zeros(d["w1"].shape, dtype=torch.float64, device="cuda")
        dw2 = torch.zeros(d["w2"].shape, dtype=torch.float64, device="cuda")
    for e in range(E):
        pr = (flat == e).nonzero().flatten()  # the expert's pairs, in order
        if not len(pr):
            continue
        t = pr // K
        w1, w2 = _fake_weight(d["w1"][e], p2), _fake_weight(d["w2"][e], p2)
        g, u, h, y = _ffn(x[t], w1, w2, p2)
        out.index_add_(0, t, wf[pr, None] * y)
        if kind != "train":
            continue
        dw[pr] = (y * dout[t]).sum(1)
        dy = _b(wf[pr, None].float() * d["dout"][t].float())
        dh = _b(_fake(dy, p2) @ w2)
        dw2[e] = _fake_cols(dy, p2).t() @ _fake_cols(_b(h), p2)
        sg = torch.sigmoid(g)
        dc = _b(torch.cat([dh * u * sg * (1 + g * (1 - sg)), dh * g * sg], 1))
        dx.index_add_(0, t, _b(_fake(dc, p2) @ w1))
        dw1[e] = _fake_cols(dc, p2).t() @ _fake_cols(d["x"][t], p2)
    if kind != "train":
        return out
    dw = dw.view(T, K)
    dp = torch.zeros_like(p).scatter_(1, idx, (dw - (dw * wk).sum(1, keepdim=True)) / pk.sum(1, keepdim=True))
    dlogits = p * (dp - (p * dp).sum(1, keepdim=True))
    return [out, dx, dlogits, dw1, dw2]
