"""Router + sort + dispatch of one batch (smoe_route_dispatch) against the
separate launches, byte for byte, on both sides of its lines (16 tokens, or 32
at up to 32 experts, routed inside, 256 tokens and 2048 pairs for the small-batch kernel),
for every router width, both scale rules, short last groups and rows longer
than the preloaded 8192 columns; and its own gating linear against float64."""
import pytest
import torch

import smoe
from smoe import ops
from smoe import workloads as W

pytestmark = pytest.mark.gpu

CASES = [
    # T, H, E, K, bias
    (1, 2048, 128, 8, False), (1, 16, 1, 1, True), (2, 144, 2, 2, False), (15, 512, 7, 3, True),
    (16, 2880, 32, 4, False), (17, 1024, 60, 6, True), (32, 4096, 8, 2, False), (33, 4096, 8, 2, True),
    (31, 7168, 256, 8, True), (64, 9232, 300, 5, False), (256, 7168, 256, 8, False), (257, 1024, 64, 4, True),
    (40, 256, 1024, 32, False), (32, 256, 32, 4, False), (32, 256, 33, 4, False), (65, 256, 40, 32, False), (128, 2048, 128, 8, False),
]


@pytest.mark.parametrize("T,H,E,K,biased", CASES)
@pytest.mark.parametrize("scale", ["amax", "pow2"])
def test_equals_separate_launches(dev, T, H, E, K, biased, scale):
    print("[dispatch]", T, H, E, K, biased, scale, flush=True)
    x = W.tokens(T, H, device=dev, outliers=True, seed=T)
    logits = W.logits(T, E, device=dev, seed=E)
    if T > 2:
        logits[1] = 0.25  # a row of ties: the lowest ids win
        logits[2, 0] = float("nan")
    bias = W.router_bias(E, device=dev) if biased else None
    got = ops.route_dispatch(x, logits, K, bias, scale=scale)
    ref = ops.route_topk_sort(logits, K, bias)
    ref += ops.permute_quant_rows(x, ref[3], K, scale=scale)
    bits = lambda t: t.contiguous().view(torch.uint8)
    for name, a, b in zip(("idx", "w", "row_map", "inv_map", "counts", "offsets", "xq", "xs"), got, ref):
        assert torch.equal(bits(a), bits(b)), name
    assert int(ops.last_route_status(dev)) == 0


@pytest.mark.parametrize("T,H,E,K", [(1, 2048, 128, 8), (3, 16, 5, 2), (32, 4096, 8, 2), (33, 2880, 32, 4),
                                     (18, 7168, 256, 8), (128, 2048, 128, 8), (100, 1040, 61, 3)])
def test_gating_linear(dev, T, H, E, K):
    """fp32 sums of H products: off from float64 by at most H * 2^-24 of the
    sum of magnitudes, so are the weights (a softmax of values of order 1)."""
    print("[gate]", T, H, E, K, flush=True)
    x = W.tokens(T, H, device=dev, seed=3)
    wg = torch.randn((H, E), generator=torch.Generator(device=dev).manual_seed(5), device=dev) * H ** -0.5
    idx, w, _, inv_map, _, offsets, xq, xs = ops.route_dispatch(x, None, K, w_gate=wg)
    l64 = x.double() @ wg.double()
    p = l64.softmax(1)
    pk, _ = p.sort(1, descending=True)
    gap = torch.cat([pk, torch.zeros_like(pk[:, :1])], 1).diff(dim=1).abs()[:, :K].amin(1)
    clear = gap > 1e-5  # no near-tie among the first K + 1
    ref_p, ref_i = p.topk(K, dim=1)
    assert torch.equal(idx[clear].long(), ref_i[clear]) and clear.float().mean() > 0.5
    ref_w = ref_p / ref_p.sum(1, keepdim=True)
    assert (w[clear].double() - ref_w[clear]).abs().max() < 1e-5
    # the rest follows from the ids
    row_map, inv, _, off = ops.route_sort(idx, E)
    q, s = ops.permute_quant_rows(x, inv, K)
    assert torch.equal(inv_map, inv) and torch.equal(offsets, off)
    assert torch.equal(xq.view(torch.uint8), q.view(torch.uint8)) and torch.equal(xs, s)


def test_layer_forms_its_logits_only_where_it_may(dev):
    m = smoe.SimpleMoE(256, 128, 8, 2, device=dev)
    m.reset_parameters(torch.Generator(device=dev).manual_seed(0))
    x = W.tokens(8, 256, device=dev)
    assert m._gate_fused(x) and not m._gate_fused(x.float()) and not m._gate_fused(x.repeat(40, 1))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not m._gate_fused(x)
    with torch.no_grad():
        a, (b, inter) = m(x), m(x, return_intermediates=True)
    xg = x.clone().requires_grad_(True)
    c = m(xg)
    assert torch.equal(a, b) and torch.equal(a, c.detach())  # the same sums in all three
    assert torch.equal(inter["logits"], ops.gate_logits(x, m.w_gate.detach(), 2))
    ref = x.double() @ m.w_gate.double()
    assert (inter["logits"] - ref).abs().max() <= 256 * 2**-24 * (x.double().abs() @ m.w_gate.double().abs()).max()
    # its gradients are those of x.float() @ w_gate
    lg = m._gate_logits(xg)
    g = torch.randn_like(lg)
    gx, gw = torch.autograd.grad(lg, (xg, m.w_gate), g)
    rx, rw = torch.autograd.grad(xg.float() @ m.w_gate, (xg, m.w_gate), g)
    assert torch.equal(gx, rx) and torch.equal(gw, rw)
