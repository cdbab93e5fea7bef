"""The layer's one-call forward and backward (smoe_layer_forward,
smoe_layer_backward) against the operators they stand for, called one by one:
every output byte for byte, over the GEMM forms (plain and packed, both
recipes), widths that are not multiples of 128, a router bias, both
weight-gradient recipes and accumulation into gradient buffers."""
import ctypes

import pytest
import torch

import smoe
from smoe import _C, ops
from smoe import workloads as W

u8 = lambda t: t.contiguous().view(torch.uint8)


def forward(m, x, logits, save):
    w1, w1s, w2, w2s = m.gemm_weights()
    rs, e8 = m._row_scale, m._pow2
    idx, w, rm, inv, cnt, off = ops.route_topk_sort(logits, m.top_k, m.router_bias)
    xq, xs = ops.permute_quant_rows(x, inv, m.top_k, scale=rs)
    st = dict(topk_idx=idx, topk_w=w, row_map=rm, inv_map=inv, counts=cnt, offsets=off, xq=xq, xs=xs)
    if save:
        st["c1"] = ops.grouped_gemm_fp8(xq, xs, w1, w1s, off, e8m0=e8)
        st["hq"], st["hs"], st["h"] = ops.swiglu_quant(st["c1"], save_h=True, scale=rs)
    else:
        st["hq"], st["hs"] = ops.grouped_gemm_fp8_swiglu(xq, xs, w1, w1s, off, scale=rs)
    st["y"] = ops.grouped_gemm_fp8(st["hq"], st["hs"], w2, w2s, off, e8m0=e8)
    return ops.unpermute_combine(st["y"], inv, w), st


def backward(m, x, logits, st, dout, dw1=None, dw2=None):
    w1t, w1ts, w2t, w2ts = m.gemm_weights_t()
    off, K, rs, e8 = st["offsets"], m.top_k, m._row_scale, m._pow2
    p2 = e8 or m.wgrad_recipe == "e8m0"
    cs = "pow2" if p2 else "fp32"
    hT, hTs, pad, ld = ops.quant_cols(st["h"], off, col_scale=cs)
    xT, xTs, _, _ = ops.quant_cols(x, off, gather=st["row_map"], gather_div=K, col_scale=cs)
    dyq, dys, dyT, dyTs, _, _, dw = ops.unpermute_combine_bwd_quant(
        dout, st["y"], st["inv_map"], st["row_map"], st["topk_w"], off, col_scale=cs, row_scale=rs)
    dw2 = ops.grouped_gemm_fp8_wgrad(dyT, dyTs, hT, hTs, pad, ld, out=dw2, accumulate=dw2 is not None, e8m0=p2)
    dh = ops.grouped_gemm_fp8(dyq, dys, w2t, w2ts, off, e8m0=e8)
    dcq, dcs, dcT, dcTs, _, _ = ops.swiglu_bwd_quant(st["c1"], dh, off, col_scale=cs, row_scale=rs)
    dw1 = ops.grouped_gemm_fp8_wgrad(dcT, dcTs, xT, xTs, pad, ld, out=dw1, accumulate=dw1 is not None, e8m0=p2)
    dxs = ops.grouped_gemm_fp8(dcq, dcs, w1t, w1ts, off, e8m0=e8)
    dx = ops.unpermute_combine(dxs, st["inv_map"], torch.ones_like(st["topk_w"]))
    return dict(dx=dx, dw1=dw1, dw2=dw2, dtopk_w=dw, dyq=dyq, dys=dys, dh=dh, dxs=dxs,
                dlogits=ops.router_topk_bwd(logits, st["topk_idx"], dw))


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,I,E,K,bias", [
    (300, 512, 512, 8, 2, False),    # packed both
    (70, 1024, 384, 4, 3, True),     # w2 plain in the default recipe
    (600, 256, 144, 4, 2, False),    # I not a multiple of 128, plain
    (257, 144, 640, 60, 8, True),    # H short, many small experts
    (1, 528, 512, 8, 1, False),
])
@pytest.mark.parametrize("recipe,wgrad", [("blockwise", "fp32"), ("blockwise", "e8m0"), ("e8m0", "fp32")])
def test_layer_calls_equal_their_operators(dev, T, H, I, E, K, bias, recipe, wgrad):
    print("[layer]", T, H, I, E, K, bias, recipe, wgrad, flush=True)
    m = smoe.SimpleMoE(H, I, E, K, device=dev, router_bias=bias, recipe=recipe, wgrad_recipe=wgrad)
    m.reset_parameters(torch.Generator(device=dev).manual_seed(T))
    if bias:
        m.router_bias.copy_(W.router_bias(E, device=dev))
    x, logits = W.tokens(T, H, device=dev), W.logits(T, E, device=dev)
    with torch.no_grad():
        out = m(x, logits)
    ref, _ = forward(m, x, logits, save=False)
    assert torch.equal(u8(out), u8(ref))
    out, st = m(x, logits, return_intermediates=True)
    ref, rst = forward(m, x, logits, save=True)
    assert torch.equal(u8(out), u8(ref))
    for k, v in rst.items():
        assert torch.equal(u8(st[k]), u8(v)), k
    dout = (W.tokens(T, H, device=dev, seed=4).float() * 1e-3).to(torch.bfloat16)
    r = backward(m, x, logits, rst, dout)
    g = m.backward_from(st, dout)
    for k, v in r.items():
        assert torch.equal(u8(g[k]), u8(v)), k
    base = torch.randn(m.w1.shape, generator=torch.Generator(device=dev).manual_seed(1), device=dev)
    b16 = torch.zeros(m.w2.shape, dtype=torch.bfloat16, device=dev) + 0.5
    r = backward(m, x, logits, rst, dout, dw1=base.clone(), dw2=b16.clone())
    g = m.backward_from(st, dout, dw1_into=base, dw2_into=b16)
    assert g["dw1"] is base and torch.equal(base, r["dw1"]) and torch.equal(b16, r["dw2"])


@pytest.mark.gpu
def test_layer_calls_refuse_what_the_operators_refused(dev):
    m = smoe.SimpleMoE(256, 128, 8, 2, device=dev)
    m.reset_parameters(torch.Generator(device=dev).manual_seed(0))
    x, lg = W.tokens(8, 256, device=dev), W.logits(8, 8, device=dev)
    with torch.no_grad():
        for bad in ((x[:, :128], lg), (x, lg[:4]), (x, lg[:, :4]), (x.cpu(), lg), (x[0], lg)):
            with pytest.raises(ValueError):
                m(*bad)
    out, st = m(x, lg, return_intermediates=True)
    with pytest.raises(ValueError):
        m.backward_from(st, x[:4])
    with pytest.raises(ValueError):
        m.backward_from(dict(st, y=st["y"][:3]), x)
    with pytest.raises(TypeError):
        m.backward_from(dict(st, c1=st["c1"].float()), x)


@pytest.mark.gpu
@pytest.mark.parametrize("recipe", ["blockwise", "e8m0"])
def test_layer_with_replaced_weights(dev, recipe):
    """Weights of other sizes put into a module run as in a module of those
    sizes (fewer experts, another width), and x wider than w2's rows as the
    operators run it (rows padded by the caller to whole 128-column groups)."""
    print("[replaced]", recipe, flush=True)
    g = torch.Generator(device=dev).manual_seed(3)
    small, m = (smoe.SimpleMoE(H, I, E, 2, device=dev, recipe=recipe) for H, I, E in ((512, 256, 4), (512, 512, 8)))
    small.reset_parameters(g)
    m.w1.data, m.w2.data, m.w_gate.data = small.w1.data, small.w2.data, small.w_gate.data
    x, lg = W.tokens(40, 512, device=dev), W.logits(40, 4, device=dev)
    with torch.no_grad():
        assert torch.equal(m(x, lg), small(x, lg)) and torch.equal(m(x), small(x))
        a, b = (q(x, lg, return_intermediates=True)[1] for q in (m, small))
        for k in ("c1", "hq", "y", "offsets"):
            assert torch.equal(u8(a[k]), u8(b[k])), k
    odd = smoe.SimpleMoE(528, 256, 4, 2, device=dev, recipe=recipe)
    odd.reset_parameters(g)
    wide = torch.nn.functional.pad(W.tokens(40, 528, device=dev), (0, 640 - 528))
    with torch.no_grad():
        out = odd(wide, lg)
        assert out.shape == (40, 528) and torch.equal(u8(out), u8(odd(wide[:, :528], lg)))
        assert torch.equal(u8(out), u8(odd(wide, lg, return_intermediates=True)[0]))


def test_layer_entry_points_reject():
    lib = _C.lib()
    assert lib.smoe_layer_forward(None, None) == -1 and lib.smoe_layer_backward(None, None, None) == -1
    fake = 0x100000
    f = _C.LayerFwd(4, 256, 128, 8, 2, 0)
    f.scratch = fake
    assert lib.smoe_layer_forward(ctypes.byref(f), None) == -5
    f.scratch = fake + 4
    assert lib.smoe_layer_forward(ctypes.byref(f), None) == -6
    f.T = 0
    assert lib.smoe_layer_forward(ctypes.byref(f), None) == -2
    b = _C.LayerBwd(4, 256, 128, 8, 2, 0)
    assert lib.smoe_layer_backward(ctypes.byref(b), None, None) == -1
    b.scratch = b.offsets = fake
    assert lib.smoe_layer_backward(ctypes.byref(b), None, None) == -5
    b.E = 5000
    assert lib.smoe_layer_backward(ctypes.byref(b), None, None) == -4
