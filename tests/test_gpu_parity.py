"""GPU parity: every HIP kernel, called through the C ABI (smoe.ops -> ctypes
-> libsmoe.so), against the CPU oracle on the same seeded inputs.

Bars: bit-exact for router ids/weights, sort maps, fp8 bytes and scales,
SwiGLU requant (given the same input) and combine; grouped-GEMM outputs
within max|d|/max|ref| <= 1e-2 and mean|d|/mean|ref| <= 1e-3 against the
float64 oracle rounded to bf16 (the reference path's output dtype).

GEMM calls of few rows per expert or few tiles run on the small-row kernel,
as most of the small shapes here do; tests/test_gpu_tile_edges.py has the edge
cases on the 256-row kernels as well, and pins which shape takes which."""
import os
import sys

import numpy as np
import pytest
import torch

from oracle import smoe_oracle as O
import smoe
from smoe import ops, workloads as W

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden")
MAX_REL, MEAN_REL = 1e-2, 1e-3


def say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


def np_u16(t):  # bf16 tensor -> uint16 numpy
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def np_u8(t):
    return t.detach().cpu().contiguous().view(torch.uint8).numpy()


def to_bf16(u16, dev):
    return torch.from_numpy(np.ascontiguousarray(u16).view(np.int16)).view(torch.bfloat16).to(dev)


def to_fp8(u8, dev):
    return torch.from_numpy(np.ascontiguousarray(u8)).view(torch.float8_e4m3fn).to(dev)


def gemm_close(got64, ref64, what=""):
    """The reference path writes bf16 (C5: fp32 accumulate, bf16 RNE store), so
    the float64 oracle is rounded to bf16 before the comparison; rounding alone
    would otherwise contribute a mean relative error of about 1.4e-3."""
    ref64 = O.bf16_to_f32(O.f32_to_bf16(np.asarray(ref64, np.float32))).astype(np.float64)
    d = np.abs(got64 - ref64)
    mx = d.max() / max(np.abs(ref64).max(), 1e-30)
    mn = d.mean() / max(np.abs(ref64).mean(), 1e-30)
    assert mx <= MAX_REL and mn <= MEAN_REL, f"{what}: max_rel={mx:.3e} mean_rel={mn:.3e}"
    return mx, mn


# ------------------------------------------------------------------ router
@pytest.mark.parametrize("T,E,K,bias", [(2048, 8, 2, False), (4096, 256, 8, True),
                                        (1024, 128, 8, False), (257, 1024, 32, True),
                                        (100, 32, 1, False)])
def test_router_bit_exact(dev, T, E, K, bias):
    say("router", T, E, K, bias)
    lg = W.logits(T, E)
    b = W.router_bias(E) if bias else None
    idx, w = ops.router_topk(lg.to(dev), K, None if b is None else b.to(dev))
    ri, rw = O.router_topk(lg.numpy(), K, None if b is None else b.numpy())
    assert np.array_equal(idx.cpu().numpy(), ri)
    assert np.array_equal(w.cpu().numpy().view(np.uint32), rw.view(np.uint32))


@pytest.mark.parametrize("T,E,K,bias", [(4096, 256, 8, True), (2048, 8, 2, False),
                                        (300, 1024, 32, False), (1000, 37, 6, True)])
def test_router_bwd_matches_oracle(dev, T, E, K, bias):
    """dlogits from the HIP router backward against the float64 oracle
    (itself pinned to torch autograd); fp32 arithmetic, so a relative bar."""
    say("router bwd", T, E, K, bias)
    lg = W.logits(T, E)
    b = W.router_bias(E) if bias else None
    idx, _ = ops.router_topk(lg.to(dev), K, None if b is None else b.to(dev))
    g = torch.randn((T, K), generator=torch.Generator().manual_seed(3))
    dl = ops.router_topk_bwd(lg.to(dev), idx, g.to(dev)).cpu().numpy().astype(np.float64)
    ref = O.router_topk_bwd(lg.numpy(), idx.cpu().numpy(), g.numpy().astype(np.float64))
    d = np.abs(dl - ref)
    assert d.max() <= 1e-5 * np.abs(ref).max(), d.max() / np.abs(ref).max()
    assert d.mean() <= 1e-6 * np.abs(ref).mean()


def test_router_ties(dev):
    say("router ties")
    rng = np.random.default_rng(11)
    lg = rng.integers(-2, 3, (512, 64)).astype(np.float32)
    idx, w = ops.router_topk(torch.from_numpy(lg).to(dev), 6)
    ri, rw = O.router_topk(lg, 6)
    assert np.array_equal(idx.cpu().numpy(), ri)
    assert np.array_equal(w.cpu().numpy(), rw)


@pytest.mark.parametrize("E,K,bias", [(256, 8, True), (256, 8, False), (64, 32, True),
                                     (16, 16, False), (1024, 32, True), (37, 32, False)])
def test_router_extremes(dev, E, K, bias):
    """Rows that reach every branch of the selection: logits spread over
    hundreds of nats (probabilities that underflow to 0 or sit below 2^-100,
    where the quotient is formed by the IEEE division), integer ties in
    logits and bias, K up to E (lanes that exhaust their candidate slots and
    rescan), rows made NaN by a NaN, a +inf or all -inf logits (ids 0..K-1
    and NaN weights, as the oracle's stable argsort gives) and a row with
    one -inf logit."""
    say("router extremes", E, K, bias)
    rng = np.random.default_rng(E * 100 + K)
    T = 256
    lg = rng.standard_normal((T, E)).astype(np.float32)
    lg[0:64] *= 60.0                                            # huge spreads
    lg[64:128] = rng.integers(-2, 3, (64, E)).astype(np.float32)  # ties
    lg[128:160] = -1e30                                         # one expert per row survives
    lg[128:160, 0] = 0.0
    lg[200] = np.nan
    lg[201, E // 3] = np.nan                                    # one NaN: the whole row is NaN
    lg[202, E // 2] = np.inf                                    # +inf: inf - inf, the row is NaN
    lg[203] = -np.inf                                           # all -inf: NaN row
    lg[204, E - 1] = -np.inf                                    # one -inf: probability 0
    b = None
    if bias:
        b = rng.integers(-1, 2, E).astype(np.float32) * np.float32(0.25)
    with np.errstate(invalid="ignore"):
        ri, rw = O.router_topk(lg, K, b)
    idx, w = ops.router_topk(torch.from_numpy(lg).to(dev), K,
                             None if b is None else torch.from_numpy(b).to(dev))
    gi, gw = idx.cpu().numpy(), w.cpu().numpy()
    assert np.array_equal(gi, ri)
    fin = ~np.isnan(rw)
    assert np.array_equal(np.isnan(gw), ~fin)
    assert np.array_equal(gw[fin].view(np.uint32), rw[fin].view(np.uint32))
    got = ops.route_topk_sort(torch.from_numpy(lg).to(dev), K,
                              None if b is None else torch.from_numpy(b).to(dev))
    assert np.array_equal(got[0].cpu().numpy(), ri)
    gw2 = got[1].cpu().numpy()
    assert np.array_equal(gw2[fin].view(np.uint32), rw[fin].view(np.uint32))


# -------------------------------------------------------------------- sort
def _check_sort(dev, idx_np, E):
    T, K = idx_np.shape
    rm, im, cnt, off = ops.route_sort(torch.from_numpy(idx_np).to(dev), E)
    r = O.route_sort(idx_np, E)
    for got, ref, n in zip((rm, im, cnt, off), r, ("row_map", "inv_map", "counts", "offsets")):
        assert np.array_equal(got.cpu().numpy(), ref), n


def test_sort_worked_example(dev):
    say("sort worked example")
    g = np.load(os.path.join(GOLDEN, "worked_example.npz"))
    _check_sort(dev, g["topk_idx"], 8)
    _, _, cnt, _ = ops.route_sort(torch.from_numpy(g["topk_idx"]).to(dev), 8)
    assert cnt.cpu().tolist() == [5, 4, 5, 4, 3, 4, 4, 3]


@pytest.mark.parametrize("T,K,E,mode", [(16384, 8, 256, "router"), (1, 1, 1, "rand"),
                                        (1, 4, 8, "rand"), (3000, 2, 8, "one"),
                                        (5000, 3, 1024, "rand"), (777, 5, 37, "skew"),
                                        (2048, 2, 8, "router")])
def test_sort_bit_exact(dev, T, K, E, mode):
    say("sort", T, K, E, mode)
    rng = np.random.default_rng(T + K + E)
    if mode == "router":
        idx = O.router_topk(W.logits(T, E).numpy(), K)[0]
    elif mode == "one":
        idx = np.full((T, K), 3, np.int32)
    elif mode == "skew":
        idx = np.minimum(rng.zipf(1.3, (T, K)) - 1, E - 1).astype(np.int32)
    else:
        idx = rng.integers(0, E, (T, K)).astype(np.int32)
    _check_sort(dev, idx, E)


@pytest.mark.parametrize("T,E,K,bias", [(16384, 256, 8, True), (16384, 128, 8, False),
                                        (8192, 8, 2, False), (2048, 8, 2, False),
                                        (1000, 37, 6, True), (333, 1024, 32, False),
                                        (700, 512, 3, True), (5, 16, 1, False),
                                        (1, 4, 4, False)])
def test_route_topk_sort_fused(dev, T, E, K, bias):
    """Router with the sort's histogram counted in the same launch: the same
    bytes as router_topk then route_sort, and both equal the oracle.  Shapes
    cover 16 and 64 lanes per token, K that does not divide the 512-pair
    segment (tokens straddling two workgroups) and the bench configs."""
    say("route_topk_sort", T, E, K, bias)
    lg = W.logits(T, E)
    b = W.router_bias(E) if bias else None
    bd = None if b is None else b.to(dev)
    got = ops.route_topk_sort(lg.to(dev), K, bd)
    ri, rw = O.router_topk(lg.numpy(), K, None if b is None else b.numpy())
    ref = (ri, rw) + tuple(O.route_sort(ri, E))
    names = ("topk_idx", "topk_w", "row_map", "inv_map", "counts", "offsets")
    for g_, r_, n in zip(got, ref, names):
        assert np.array_equal(g_.cpu().numpy().view(np.uint32), np.asarray(r_).view(np.uint32)), n
    assert int(ops.last_route_status().item()) == 0


def test_route_sort_out_of_range_ids(dev):
    """Ids outside [0, E) get no row: inv_map = -1, offsets[E] counts only the
    valid pairs, the valid pairs keep the stable order, and the status word
    holds the number dropped; check_route_status raises on it."""
    say("route_sort out-of-range ids")
    T, K, E = 3000, 4, 16
    rng = np.random.default_rng(7)
    idx = rng.integers(0, E, (T, K)).astype(np.int32)
    bad = rng.random((T, K)) < 0.01
    idx[bad] = rng.choice(np.array([E, E + 3, 19, -1, 1 << 20], np.int32), bad.sum())
    rm, im, cnt, off = ops.route_sort(torch.from_numpy(idx).to(dev), E)
    flat = idx.reshape(-1)
    valid = (flat >= 0) & (flat < E)
    p_valid = np.nonzero(valid)[0]
    order = p_valid[np.argsort(flat[p_valid], kind="stable")]
    nv = order.size
    assert int(ops.last_route_status().item()) == flat.size - nv
    with pytest.raises(ValueError):
        ops.check_route_status()
    im_np = im.cpu().numpy()
    assert np.all(im_np[~valid] == -1)
    assert np.array_equal(rm.cpu().numpy()[:nv], order)
    assert np.array_equal(im_np[order], np.arange(nv))
    assert np.array_equal(cnt.cpu().numpy(), np.bincount(flat[valid], minlength=E))
    assert off.cpu().numpy()[-1] == nv
    # the dropped pairs contribute nothing to the combine
    H = 128
    y = torch.randn((T * K, H), device=dev).to(torch.bfloat16)
    w = torch.ones((T, K), device=dev)
    out = ops.unpermute_combine(y, im, w).float().cpu().numpy()
    yv = y.float().cpu().numpy()
    ref = np.zeros((T, H), np.float32)
    for t in range(T):
        for k in range(K):
            r = im_np[t * K + k]
            if r >= 0:
                ref[t] = ref[t] + yv[r]
    assert np.array_equal(O.f32_to_bf16(ref), np_u16(torch.from_numpy(out).to(torch.bfloat16)))
    # a clean sort afterwards clears the status
    ops.route_sort(torch.from_numpy(np.where(valid.reshape(T, K), idx, 0)).to(dev), E)
    ops.check_route_status()


# ---------------------------------------------------------- permute_quant
def test_permute_quant_every_bf16_value(dev):
    """Each group holds one +-448 element so s == 1 and q = e4m3(x): every
    finite bf16 value with |x| <= 448 passes through the GPU encoder."""
    say("permute_quant exhaustive bf16")
    u = np.arange(1 << 16, dtype=np.uint32)
    v = (u << 16).view(np.float32)
    v = v[np.isfinite(v) & (np.abs(v) <= 448)]
    n = -(-v.size // 127) * 127
    vals = np.zeros(n, np.float32)
    vals[:v.size] = v
    rows = vals.reshape(-1, 127)
    x = np.concatenate([np.full((rows.shape[0], 1), 448.0, np.float32), rows], axis=1)
    x = x.reshape(-1, 1024) if x.size % 1024 == 0 else x.reshape(-1, 128)
    xb = O.f32_to_bf16(x)
    T = xb.shape[0]
    inv = np.arange(T, dtype=np.int32)
    xq, xs = ops.permute_quant_rows(to_bf16(xb, dev), torch.from_numpy(inv).to(dev), 1)
    rq, rs = O.permute_quant(xb, inv, 1)
    assert np.array_equal(np_u8(xq), rq)
    assert np.array_equal(xs.cpu().numpy(), rs)
    assert (rs == 1.0).all()


def test_fast_quantiser_exhaustive(dev):
    """The bf16 kernels (permute, row, column and weight quantisation) divide
    by the group scale with a reciprocal and one residual correction instead
    of an IEEE division, and every kernel encodes with the hardware fp8
    conversion instead of the software RNE encoder.  The library's self-test
    compares both with the reference rule exhaustively: every finite bf16 x
    against every positive finite bf16 amax >= |x| (s = amax / 448), and every
    fp32 with |v| <= 448 through the encoder.  The bf16 outputs (GEMM
    epilogue, combine, SwiGLU h, backward) use the hardware fp32 -> bf16
    conversion, checked against the software RNE rule for all 2^32 fp32
    patterns."""
    say("fast quantiser exhaustive")
    counts = torch.zeros(6, dtype=torch.int64, device=dev)
    smoe._C.call("smoe_selftest_quant", counts.data_ptr(), torch.cuda.current_stream().cuda_stream)
    bad_div, n_div, bad_enc, n_enc, bad_bf, n_bf = counts.cpu().tolist()
    assert n_div == sum(2 * (a + 1) for a in range(1, 0x7f80))
    assert n_enc == 2 * (0x43e00000 + 1)
    assert n_bf == 2 * 2**32
    assert bad_div == 0 and bad_enc == 0 and bad_bf == 0


def test_reciprocal_exhaustive(dev):
    """The SwiGLU backward's sigmoid forms 1/b as v_rcp_f32 plus one Newton
    step instead of an IEEE division.  The library's self-test compares the
    two for every fp32 b in [2^-126, 2^126) and for +inf: no mismatch."""
    say("reciprocal exhaustive")
    counts = torch.zeros(2, dtype=torch.int64, device=dev)
    smoe._C.call("smoe_selftest_recip", counts.data_ptr(), torch.cuda.current_stream().cuda_stream)
    bad, n = counts.cpu().tolist()
    assert n == 252 * 2**23 + 1
    assert bad == 0


@pytest.mark.parametrize("T,H,E,K,outl", [(2048, 1024, 8, 2, False), (1024, 7168, 256, 8, True),
                                          (333, 4096, 8, 2, False), (512, 2048, 128, 8, False),
                                          (5, 1152, 4, 3, True), (64, 9216, 16, 4, True),
                                          # rows split over two waves: 5 chunks (the second wave's
                                          # last chunk past the row, one of its groups live), 6, 8,
                                          # and an odd T (a block's last waves past the tokens)
                                          (7, 4224, 16, 3, True), (9, 6144, 8, 2, False),
                                          (130, 8192, 64, 8, True), (3, 7168, 256, 8, True)])
def test_permute_quant_bit_exact(dev, T, H, E, K, outl):
    say("permute_quant", T, H, E, K, outl)
    x = W.tokens(T, H, outliers=outl)
    lg = W.logits(T, E)
    idx = O.router_topk(lg.numpy(), K)[0]
    xq, xs, rm, im, cnt, off = ops.permute_quant(x.to(dev), torch.from_numpy(idx).to(dev), E)
    r_rm, r_im, r_cnt, r_off = O.route_sort(idx, E)
    assert np.array_equal(rm.cpu().numpy(), r_rm) and np.array_equal(im.cpu().numpy(), r_im)
    assert np.array_equal(off.cpu().numpy(), r_off) and np.array_equal(cnt.cpu().numpy(), r_cnt)
    rq, rs = O.permute_quant(np_u16(x), r_im, K)
    assert np.array_equal(np_u8(xq), rq)
    assert np.array_equal(xs.cpu().numpy().view(np.uint32), rs.view(np.uint32))


@pytest.mark.parametrize("T,K,E,mode", [(1000, 3, 16, "rand"), (700, 6, 64, "skew"),
                                        (300, 7, 1024, "rand"), (160, 32, 64, "rand"),
                                        (2000, 5, 8, "one"), (1, 1, 1, "rand"),
                                        (4099, 8, 256, "skew")])
def test_dispatch_matches_sort(dev, T, K, E, mode):
    """smoe_dispatch_quant end to end.  K values that do not divide the
    512-pair sort segment make tokens straddle segments; skewed and
    single-expert loads stress the per-expert scan.  Maps, counts, offsets,
    fp8 bytes and scales must equal the oracle's sort + permute."""
    say("dispatch", T, K, E, mode)
    rng = np.random.default_rng(T * K + E)
    if mode == "one":
        idx = np.full((T, K), E - 1, np.int32)
    elif mode == "skew":
        idx = np.minimum(rng.zipf(1.2, (T, K)) - 1, E - 1).astype(np.int32)
    else:
        idx = rng.integers(0, E, (T, K)).astype(np.int32)
    H = 256
    x = W.tokens(T, H, outliers=True)
    xq, xs, rm, im, cnt, off = ops.permute_quant(x.to(dev), torch.from_numpy(idx).to(dev), E)
    r_rm, r_im, r_cnt, r_off = O.route_sort(idx, E)
    for got, ref, n in zip((rm, im, cnt, off), (r_rm, r_im, r_cnt, r_off),
                           ("row_map", "inv_map", "counts", "offsets")):
        assert np.array_equal(got.cpu().numpy(), ref), n
    rq, rs = O.permute_quant(np_u16(x), r_im, K)
    assert np.array_equal(np_u8(xq), rq)
    assert np.array_equal(xs.cpu().numpy().view(np.uint32), rs.view(np.uint32))


def test_permute_quant_zero_and_saturating_groups(dev):
    say("permute_quant zero/sat groups")
    T, H = 8, 256
    x = np.zeros((T, H), np.float32)
    x[1, :] = 3.0e38                         # bf16 near max: s large, all 448
    x[2, 5] = -1e-40                         # denormal-range input
    x[3, ::2] = 1.0
    x[3, 1::2] = -2.0 ** -20                 # tiny values flush to +-0 codes
    xb = O.f32_to_bf16(x)
    inv = np.arange(T, dtype=np.int32)
    xq, xs = ops.permute_quant_rows(to_bf16(xb, dev), torch.from_numpy(inv).to(dev), 1)
    rq, rs = O.permute_quant(xb, inv, 1)
    assert np.array_equal(np_u8(xq), rq) and np.array_equal(xs.cpu().numpy(), rs)
    assert (rs[0] == 1.0).all()


def test_non_finite_groups_stay_local(dev):
    """A 128-wide group holding a NaN or +-inf has unspecified bytes (the
    quantisation rule is for finite inputs), but the kernels run through it
    and every finite group, in the same row or elsewhere, keeps its exact
    bytes and scale: permute_quant, row quantisation and the SwiGLU
    requantisation."""
    say("non-finite groups")
    rng = np.random.default_rng(21)
    T, H, K = 64, 1024, 2
    x = rng.standard_normal((T, H)).astype(np.float32)
    x[3, 5], x[7, 300], x[9, 1000], x[11, :128] = np.nan, np.inf, -np.inf, np.nan
    xb = O.f32_to_bf16(x)
    bad = ~np.isfinite(O.bf16_to_f32(xb)).reshape(T, H // 128, 128).all(axis=2)  # [T, groups]
    idx = np.stack([rng.permutation(8)[:K] for _ in range(T)]).astype(np.int32)
    rm, im, _, _ = O.route_sort(idx, 8)
    xq, xs = ops.permute_quant_rows(to_bf16(xb, dev), torch.from_numpy(im).to(dev), K)
    xf = np.where(np.repeat(bad, 128, axis=1), np.float32(0), O.bf16_to_f32(xb))
    rq, rs = O.permute_quant(O.f32_to_bf16(xf), im, K)
    ok = ~bad[rm // K]                                   # [R, groups] of finite groups
    gq = np_u8(xq).reshape(-1, H // 128, 128)
    assert np.array_equal(gq[ok], rq.reshape(-1, H // 128, 128)[ok])
    assert np.array_equal(xs.cpu().numpy()[ok], rs[ok])
    q, s = ops.quant_rows(to_bf16(xb, dev))
    rq2, rs2 = O.quant_1x128(xf)
    assert np.array_equal(np_u8(q).reshape(T, -1, 128)[~bad], rq2.reshape(T, -1, 128)[~bad])
    assert np.array_equal(s.cpu().numpy()[~bad], rs2[~bad])
    # SwiGLU: c1 = [g | u] with non-finite values in a few g and u groups
    c1 = rng.standard_normal((T, 2 * H)).astype(np.float32)
    c1[2, 7], c1[4, H + 200], c1[6, 600] = np.nan, np.inf, -np.inf
    cb = O.f32_to_bf16(c1)
    hq, hs = ops.swiglu_quant(to_bf16(cb, dev))
    cf = O.bf16_to_f32(cb)
    hbad = ~(np.isfinite(cf[:, :H]) & np.isfinite(cf[:, H:])).reshape(T, H // 128, 128).all(axis=2)
    cf = np.where(np.repeat(np.concatenate([hbad, hbad], axis=1), 128, axis=1), np.float32(0), cf)
    rhq, rhs = O.swiglu_quant(O.f32_to_bf16(cf))
    assert np.array_equal(np_u8(hq).reshape(T, -1, 128)[~hbad], rhq.reshape(T, -1, 128)[~hbad])
    assert np.array_equal(hs.cpu().numpy()[~hbad], rhs[~hbad])


def test_permute_quant_config2_full(dev):
    """Benchmark config 2 at full size (T=16384, H=7168, E=256, top-8, bias,
    outliers): ids, maps, counts, fp8 bytes and scales all bit-exact."""
    say("permute_quant config2 full")
    c = W.CONFIGS["permute"]
    x = W.tokens(c.T, c.H, outliers=True)
    lg, b = W.logits(c.T, c.E), W.router_bias(c.E)
    idx, w = ops.router_topk(lg.to(dev), c.K, b.to(dev))
    ri, rw = O.router_topk(lg.numpy(), c.K, b.numpy())
    assert np.array_equal(idx.cpu().numpy(), ri)
    xq, xs, rm, im, cnt, off = ops.permute_quant(x.to(dev), idx, c.E)
    r_rm, r_im, r_cnt, r_off = O.route_sort(ri, c.E)
    assert np.array_equal(rm.cpu().numpy(), r_rm)
    assert np.array_equal(off.cpu().numpy(), r_off)
    rq, rs = O.permute_quant(np_u16(x), r_im, c.K)
    assert np.array_equal(np_u8(xq), rq)
    assert np.array_equal(xs.cpu().numpy(), rs)


# ------------------------------------------------------------- weights
def test_weight_quant_golden_and_random(dev):
    say("weight quant")
    g = np.load(os.path.join(GOLDEN, "weight_quant.npz"))
    wq, ws = ops.quantize_weight_blockwise(to_bf16(g["w"], dev))
    assert np.array_equal(np_u8(wq), g["wq"]) and np.array_equal(ws.cpu().numpy(), g["ws"])
    w = W.weights(3, 384, 640, seed=7)
    wq, ws = ops.quantize_weight_blockwise(w.to(dev))
    rq, rs = O.quantize_weight_blockwise(np_u16(w))
    assert np.array_equal(np_u8(wq), rq) and np.array_equal(ws.cpu().numpy(), rs)


# ------------------------------------------------------------------ GEMM
def _fp8_operands(rng, R, N, Kd, E):
    x = rng.standard_normal((R, Kd)).astype(np.float32)
    xq, xs = O.quant_1x128(x)
    w = O.f32_to_bf16((rng.standard_normal((E, N, Kd)) * 0.02).astype(np.float32))
    wq, ws = O.quantize_weight_blockwise(w)
    return xq, xs, wq, ws


def _run_gemm(dev, xq, xs, wq, ws, off):
    args = (to_fp8(xq, dev), torch.from_numpy(xs).to(dev), to_fp8(wq, dev),
            torch.from_numpy(ws).to(dev), torch.from_numpy(off).to(dev))
    out = ops.grouped_gemm_fp8(*args)
    E, N, Kd = wq.shape
    if ops.packed_gemm_ok(N, Kd):
        # the packed-weight kernel must give the same bytes on every row that
        # exactly one expert's range covers (malformed offsets can give a row
        # to two experts, whose writes race, or to none).  For these seeded
        # operands (quantised N(0,1) rows, N(0,0.02) weights, one-hot values)
        # every K block's products sum without rounding in the MFMA, so the
        # two kernels' K orders cannot show (tests/test_gpu_large.py has
        # operands where they do).
        got = ops.grouped_gemm_fp8(args[0], args[1], ops.pack_weight_fp8(args[2]), *args[3:])
        R = xq.shape[0]
        cover = np.zeros(R, np.int32)
        for e in range(E):
            cover[max(int(off[e]), 0):max(min(int(off[e + 1]), R), 0)] += 1
        one = torch.from_numpy(cover == 1).to(dev)
        assert torch.equal(got[one].view(torch.int16), out[one].view(torch.int16)), "packed != plain"
    return O.bf16_to_f32(np_u16(out)).astype(np.float64)


@pytest.mark.parametrize("Kd", [256, 512])
def test_gemm_layout_one_hot(dev, Kd):
    """Structured operands expose any row/column/K permutation in the MFMA
    fragment or output layout: x[r] = e_(r mod Kd), w[n] = e_n (Kd = 512 also
    runs on packed weights)."""
    say("gemm one-hot layout", Kd)
    R, N, E = 300, 256, 1
    xq = np.zeros((R, Kd), np.uint8)
    xq[np.arange(R), np.arange(R) % Kd] = 0x38  # 1.0
    xs = np.ones((R, Kd // 128), np.float32)
    wq = np.zeros((E, N, Kd), np.uint8)
    wq[0, np.arange(N), np.arange(N)] = 0x38
    ws = np.ones((E, N // 128, Kd // 128), np.float32)
    off = np.array([0, R], np.int32)
    got = _run_gemm(dev, xq, xs, wq, ws, off)
    ref = O.grouped_gemm_fp8(xq, xs, wq, ws, off)
    bad = np.argwhere(got != ref)
    assert bad.size == 0, f"{len(bad)} mismatches, first (r,n): {bad[:8].tolist()}"


@pytest.mark.parametrize("Kd", [384, 512, 1536, 3072])
def test_gemm_scale_indexing(dev, Kd):
    """Distinct scales per (row, K block) and per (expert, n block, K block).
    Kd = 384 reads the activation scales one K block at a time; the others
    stage them 8 K blocks at a time: 512 (one chunk, its second half past the
    row end), 1536 (two chunks, the last one half full) and 3072 (3 chunks:
    both halves of the chunk buffer and a reuse)."""
    say("gemm scale indexing", Kd)
    rng = np.random.default_rng(21)
    R, N, E = 200, 384, 2
    xq, xs, wq, ws = _fp8_operands(rng, R, N, Kd, E)
    xs = rng.random(xs.shape).astype(np.float32) + 0.5      # distinct per (r, kb)
    ws = rng.random(ws.shape).astype(np.float32) + 0.5      # distinct per (e, nb, kb)
    off = np.array([0, 77, R], np.int32)
    got = _run_gemm(dev, xq, xs, wq, ws, off)
    gemm_close(got, O.grouped_gemm_fp8(xq, xs, wq, ws, off), "scales")


@pytest.mark.parametrize("counts,N,Kd", [([5, 0, 300, 1, 0, 129, 128, 17], 256, 512),
                                         ([0, 0, 1000], 512, 1024),
                                         ([1], 128, 128),
                                         ([4096, 0, 0, 3], 1024, 2048),
                                         ([700, 0, 33, 1], 384, 3072)])
def test_gemm_skewed_experts(dev, counts, N, Kd):
    say("gemm skewed", counts, N, Kd)
    rng = np.random.default_rng(sum(counts) + N)
    E, R = len(counts), sum(counts)
    xq, xs, wq, ws = _fp8_operands(rng, R, N, Kd, E)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    got = _run_gemm(dev, xq, xs, wq, ws, off)
    gemm_close(got, O.grouped_gemm_fp8(xq, xs, wq, ws, off), f"{counts}")


def test_gemm_max_experts(dev):
    """E = 1024 (the maximum): the tile search covers 16 experts per lane (the
    small-row kernel), many experts own no rows, the rest own 1..300."""
    say("gemm 1024 experts")
    rng = np.random.default_rng(1024)
    E, N, Kd = 1024, 256, 256
    counts = rng.integers(0, 40, E)
    counts[rng.choice(E, 300, replace=False)] = 0
    counts[5], counts[1023] = 300, 1
    R = int(counts.sum())
    xq, xs, wq, ws = _fp8_operands(rng, R, N, Kd, E)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    got = _run_gemm(dev, xq, xs, wq, ws, off)
    gemm_close(got, O.grouped_gemm_fp8(xq, xs, wq, ws, off), "E=1024")


def test_gemm_max_kdim(dev):
    """Kdim = 65536 (the maximum): 512 K blocks, eight windows of weight scales
    in the small-row kernel."""
    say("gemm Kdim 65536")
    rng = np.random.default_rng(65536)
    counts = [3, 130]
    E, N, Kd = len(counts), 256, 65536
    R = sum(counts)
    xq, xs, wq, ws = _fp8_operands(rng, R, N, Kd, E)
    xs = (rng.random(xs.shape) + 0.5).astype(np.float32)
    ws = (rng.random(ws.shape) + 0.5).astype(np.float32)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    got = _run_gemm(dev, xq, xs, wq, ws, off)
    gemm_close(got, O.grouped_gemm_fp8(xq, xs, wq, ws, off), "Kdim=65536")


@pytest.mark.parametrize("Kd", [256, 512])
def test_gemm_malformed_offsets_stay_in_range(dev, Kd):
    """offsets[] lives on the device and is not validated on the host, so the
    kernel clamps every tile to rows [0, R): here expert 1's offsets decrease
    (no tiles) and expert 2's run past R.  No access leaves the buffers; the
    rows that belong to one expert only match the oracle.  (Kd = 512 also runs
    the packed-weight kernel, which must give the same bytes.)"""
    say("gemm malformed offsets", Kd)
    rng = np.random.default_rng(77)
    R, N, E = 1000, 256, 3
    xq, xs, wq, ws = _fp8_operands(rng, R, N, Kd, E)
    bad = np.array([0, 400, 300, 1500], np.int32)
    got = _run_gemm(dev, xq, xs, wq, ws, bad)
    ref0 = O.grouped_gemm_fp8(xq, xs, wq, ws, np.array([0, 300, 300, 300], np.int32))
    ref2 = O.grouped_gemm_fp8(xq, xs, wq, ws, np.array([0, 0, 0, R], np.int32))
    gemm_close(got[:300], ref0[:300], "expert 0 rows")
    gemm_close(got[400:], ref2[400:], "expert 2 rows, clamped at R")


def test_gemm_dsv3_shape_sampled_rows(dev):
    """Benchmark config 4 at full size (R=65536, 32 experts, Zipf loads with
    zero-token experts, fc1 N=4096 K=7168 and fc2 N=7168 K=2048); the oracle
    checks a sample of rows from every non-empty expert."""
    say("gemm dsv3 full")
    c = W.CONFIGS["dsv3"]
    counts = W.zipf_counts()
    off = W.offsets_from_counts(counts)
    x = W.tokens(c.T, c.H, device=dev)
    inv = torch.arange(c.T, dtype=torch.int32, device=dev)
    xq, xs = ops.permute_quant_rows(x, inv, 1)
    offs = off.numpy()
    rows = np.concatenate([np.unique(np.linspace(offs[e], offs[e + 1] - 1, 6).astype(np.int64))
                           for e in range(c.E) if counts[e] > 0])
    for N, Kd, seed in ((2 * c.I, c.H, 3), (c.H, c.I, 13)):
        w = W.weights(c.E, N, Kd, device=dev, seed=seed)
        wq, ws = ops.quantize_weight_blockwise(w)
        del w
        a_q, a_s = (xq, xs) if Kd == c.H else ops.permute_quant_rows(
            W.tokens(c.T, Kd, device=dev, seed=17), inv, 1)
        out = ops.grouped_gemm_fp8(a_q, a_s, wq, ws, off.to(dev))
        got = O.bf16_to_f32(np_u16(out[torch.from_numpy(rows).to(dev)])).astype(np.float64)
        aq_np, as_np = np_u8(a_q[torch.from_numpy(rows).to(dev)]), a_s[torch.from_numpy(rows).to(dev)].cpu().numpy()
        wq_np, ws_np = np_u8(wq), ws.cpu().numpy()
        ref = np.zeros_like(got)
        owner = np.searchsorted(offs, rows, side="right") - 1
        for e in np.unique(owner):
            sel = owner == e
            ref[sel] = O.dequant_rows(aq_np[sel], as_np[sel]) @ O.dequant_weight(wq_np[e], ws_np[e]).T
        gemm_close(got, ref, f"dsv3 N={N} K={Kd}")
        del wq, ws, out
        torch.cuda.empty_cache()


# ---------------------------------------------------------------- SwiGLU
@pytest.mark.parametrize("R,I", [(1000, 2048), (77, 768), (300, 128), (16, 14336), (9, 1152)])
def test_swiglu_quant_bit_exact(dev, R, I):
    say("swiglu", R, I)
    rng = np.random.default_rng(R + I)
    c1 = O.f32_to_bf16((rng.standard_normal((R, 2 * I)) * 4).astype(np.float32))
    c1[0, :8] = O.f32_to_bf16(np.array([0, 100, -100, 88.5, -88.5, -87.2, 1e-30, -0.0], np.float32))
    hq, hs = ops.swiglu_quant(to_bf16(c1, dev))
    rq, rs = O.swiglu_quant(c1)
    assert np.array_equal(np_u8(hq), rq)
    assert np.array_equal(hs.cpu().numpy().view(np.uint32), rs.view(np.uint32))


# --------------------------------------------------------------- combine
@pytest.mark.parametrize("T,K,H", [(2048, 2, 1024), (1000, 8, 7168), (3, 1, 128), (17, 5, 1152),
                                   (200, 16, 256), (77, 32, 384)])
def test_combine_bit_exact(dev, T, K, H):
    say("combine", T, K, H)
    rng = np.random.default_rng(T * K + H)
    y = O.f32_to_bf16(rng.standard_normal((T * K, H)).astype(np.float32))
    inv = rng.permutation(T * K).astype(np.int32)
    w = rng.random((T, K)).astype(np.float32)
    out = ops.unpermute_combine(to_bf16(y, dev), torch.from_numpy(inv).to(dev), torch.from_numpy(w).to(dev))
    ref = O.unpermute_combine(y, inv, w, K)
    assert np.array_equal(np_u16(out), ref)


def test_combine_identity_bytes(dev):
    say("combine identity")
    rng = np.random.default_rng(5)
    y = O.f32_to_bf16(rng.standard_normal((512, 256)).astype(np.float32))
    inv = rng.permutation(512).astype(np.int32)
    out = ops.unpermute_combine(to_bf16(y, dev), torch.from_numpy(inv).to(dev),
                                torch.ones((512, 1), dtype=torch.float32, device=dev))
    assert np.array_equal(np_u16(out), y[inv])


# ----------------------------------------------------------- whole layer
def test_layer_golden_fixture_stagewise(dev):
    """The committed tiny fixture through every kernel, stage by stage, each
    stage fed the oracle's previous-stage output."""
    say("layer golden stagewise")
    g = np.load(os.path.join(GOLDEN, "oracle_tiny.npz"))
    K, E = int(g["K"]), g["w1q"].shape[0]
    idx, w = ops.router_topk(torch.from_numpy(g["logits"]).to(dev), K)
    assert np.array_equal(idx.cpu().numpy(), g["topk_idx"]) and np.array_equal(w.cpu().numpy(), g["topk_w"])
    xq, xs, rm, im, cnt, off = ops.permute_quant(to_bf16(g["x"], dev), idx, E)
    for t, k in ((rm, "row_map"), (im, "inv_map"), (cnt, "counts"), (off, "offsets"), (xs, "xs")):
        assert np.array_equal(t.cpu().numpy(), g[k]), k
    assert np.array_equal(np_u8(xq), g["xq"])
    w1q, w1s = to_fp8(g["w1q"], dev), torch.from_numpy(g["w1s"]).to(dev)
    c1 = ops.grouped_gemm_fp8(xq, xs, w1q, w1s, off)
    gemm_close(O.bf16_to_f32(np_u16(c1)).astype(np.float64), O.bf16_to_f32(g["c1"]).astype(np.float64), "fc1")
    hq, hs = ops.swiglu_quant(to_bf16(g["c1"], dev))
    assert np.array_equal(np_u8(hq), g["hq"]) and np.array_equal(hs.cpu().numpy(), g["hs"])
    y = ops.grouped_gemm_fp8(to_fp8(g["hq"], dev), torch.from_numpy(g["hs"]).to(dev),
                             to_fp8(g["w2q"], dev), torch.from_numpy(g["w2s"]).to(dev), off)
    gemm_close(O.bf16_to_f32(np_u16(y)).astype(np.float64), O.bf16_to_f32(g["y"]).astype(np.float64), "fc2")
    out = ops.unpermute_combine(to_bf16(g["y"], dev), im, w)
    assert np.array_equal(np_u16(out), g["out"])


def test_simple_moe_config1_end_to_end(dev):
    """Benchmark config 1 (T=2048, H=1024, E=8, top-2, I=2048) through
    SimpleMoE.forward vs the oracle's whole layer on the same fp8 weights."""
    say("SimpleMoE config1")
    c = W.CONFIGS["tiny"]
    m = smoe.SimpleMoE(c.H, c.I, c.E, c.K, device=dev)
    with torch.no_grad():
        m.w1.copy_(W.weights(c.E, 2 * c.I, c.H).to(dev))
        m.w2.copy_(W.weights(c.E, c.H, c.I, seed=13).to(dev))
    x, lg = W.tokens(c.T, c.H), W.logits(c.T, c.E)
    out, st = m(x.to(dev), lg.to(dev), return_intermediates=True)
    w1q, w1s, w2q, w2s = m.fp8_weights()
    r = O.moe_forward(np_u16(x), lg.numpy(), np_u8(w1q), w1s.cpu().numpy(), np_u8(w2q),
                      w2s.cpu().numpy(), c.K)
    for k in ("topk_idx", "topk_w", "row_map", "inv_map", "offsets", "xs"):
        assert np.array_equal(st[k].cpu().numpy(), r[k]), k
    assert np.array_equal(np_u8(st["xq"]), r["xq"])
    f = lambda u: O.bf16_to_f32(u).astype(np.float64)
    gemm_close(f(np_u16(st["c1"])), f(r["c1"]), "fc1")
    # downstream of fc1 the fp8 requant may flip an ulp where c1 differs in
    # its last bf16 bit; the layer output is held to the GEMM tolerance
    gemm_close(f(np_u16(out)), f(r["out"]), "layer out")


def test_simple_moe_empty_batch(dev):
    """T = 0 tokens: the layer returns [0, H] without launching a kernel (the
    C ABI refuses T = 0), under autograd the weight gradients are zeros, and
    a normal batch right after still matches the no-autograd forward."""
    say("SimpleMoE empty batch")
    H, I, E, K = 256, 256, 8, 2
    m = smoe.SimpleMoE(H, I, E, K, device=dev)
    m.reset_parameters(torch.Generator(device=dev).manual_seed(3))
    x0 = torch.empty((0, H), dtype=torch.bfloat16, device=dev)
    with torch.no_grad():
        out = m(x0)
    assert out.shape == (0, H) and out.dtype == torch.bfloat16
    out, st = m(x0, return_intermediates=True)
    assert out.shape == (0, H) and st["offsets"].shape == (E + 1,)
    assert int(st["offsets"].abs().sum()) == 0 and st["xq"].shape == (0, H)
    g = m.backward_from(st, torch.empty((0, H), dtype=torch.bfloat16, device=dev))
    assert g["dx"].shape == (0, H) and g["dlogits"].shape == (0, E)
    assert not g["dw1"].any() and not g["dw2"].any() and not g["dw_gate"].any()
    xg = x0.clone().requires_grad_(True)
    m(xg).float().sum().backward()
    assert xg.grad.shape == (0, H)
    assert not m.w1.grad.any() and not m.w2.grad.any() and not m.w_gate.grad.any()
    x = W.tokens(64, H).to(dev)
    with torch.no_grad():
        ref = m(x)
    again = m(x)
    assert torch.equal(ref.view(torch.int16), again.detach().view(torch.int16))
