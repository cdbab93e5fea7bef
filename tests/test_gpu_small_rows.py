"""The grouped GEMM for few rows per expert (smoe_gemm_small.hip) against the
256-row kernels, byte for byte: the same operands with unused rows past
offsets[E], which push the average over every line, take the general path.
The row counts sit on the edges of the 16-row blocks and of the 112 and 128-row tiles,
K on both sides of the load-ahead and of the 64-step scale window, N on
partial column tiles; more than 256 experts take the tile search's long
form.  A CPU model checks the tile mapping for valid and malformed offsets."""
import numpy as np
import pytest
import torch

from oracle import smoe_oracle as O
from smoe import _C, ops
from smoe import workloads as W



# ------------------------------------------------------------- CPU model
def tiles(R, NT, offsets, BM):
    """(expert, first row, rows, column tile) of every workgroup that works."""
    E = len(offsets) - 1
    offsets = np.clip(offsets, 0, R)
    n = [max(0, int(offsets[e + 1]) - int(offsets[e])) for e in range(E)]
    bound = min(E, R) + -(-R // BM)
    cut64 = -(-R // 64)
    low = R > 64 and cut64 * NT <= 512  # 64-row tiles, if they all run at once
    if low:
        bound = max(bound, min(min(E, R) + cut64, -(-512 // NT)))
    cnt = [min(-(-m // BM), bound) for m in n]
    total = 0
    for b in range(0, E, 64):
        total = min(total + sum(cnt[b:b + 64]), bound)
    cnt64 = [-(-m // 64) for m in n]
    if low and sum(cnt64) * NT <= 512 and not (total * NT <= 256 < sum(cnt64) * NT):
        BM, cnt, total = 64, cnt64, sum(cnt64)
    out, n = [], total * NT
    chunk = (n + 7) // 8
    for bid in range((bound * NT + 7) // 8 * 8):
        tl = (bid & 7) * chunk + (bid >> 3)
        if (bid >> 3) >= chunk or tl >= n:
            continue
        mt, first, e = tl // NT, 0, 0
        while e < E and first + cnt[e] <= mt:
            first += cnt[e]
            e += 1
        if e == E:
            continue
        q = tl - first * NT
        nt = q // cnt[e]
        o0, o1 = int(offsets[e]), int(offsets[e + 1])
        h = min((-(-(o1 - o0) // cnt[e]) + 15) & ~15, BM)
        row0 = o0 + (q - nt * cnt[e]) * h
        rows = min(h, o1 - row0)
        if rows > 0:
            out.append((e, row0, rows, nt))
    return out


def test_tiles_cover_every_row_once():
    rng = np.random.default_rng(3)
    for _ in range(200):
        E = int(rng.integers(1, 300))
        counts = rng.integers(0, rng.choice([2, 40, 400]), E)
        counts[rng.random(E) < 0.3] = 0
        lead = int(rng.integers(0, 5))
        R = max(1, lead + int(counts.sum()) + int(rng.integers(0, 50)))
        off = lead + np.concatenate([[0], np.cumsum(counts)])
        NT = int(rng.integers(1, 4))
        seen = np.zeros((R, NT), int)
        BM = int(rng.choice([112, 128]))
        for e, row0, rows, nt in tiles(R, NT, off, BM):
            assert off[e] <= row0 and row0 + rows <= off[e + 1] and rows <= BM
            seen[row0:row0 + rows, nt] += 1
        assert (seen[off[0]:off[-1]] == 1).all() and seen.sum() == int(counts.sum()) * NT


def test_tiles_stay_in_range_for_malformed_offsets():
    rng = np.random.default_rng(4)
    for _ in range(200):
        E, R = int(rng.integers(1, 9)), int(rng.integers(1, 400))
        off = int(rng.integers(-300, 300)) + np.concatenate([[0], np.cumsum(rng.integers(-300, 900, E))])
        for _, row0, rows, _ in tiles(R, 2, off, 112):
            assert 0 <= row0 and row0 + rows <= R and rows <= 112


# loads on the edges of the choice of 64-row tiles: counts, N of the fused
# SwiGLU form (128 columns a tile), tile rows chosen
CUT = [
    ([65] * 3, 256, 64),
    ([129] * 50, 1024, 112),        # 64-row tiles: 600 workgroups, past 512; 400 of 112 rows
    ([129] * 42 + [1], 1024, 64),   # 127 x 4 workgroups
    ([128] * 64, 1024, 64),         # 128 x 4: 512 exactly
    ([128] * 63 + [129], 1024, 112),
    ([112] * 16, 4096, 112),        # 16 x 16: a CU each; the low tiles would be 512
    ([113] + [112] * 15, 4096, 64),
    ([113, 113] + [40] * 13, 4096, 64),
    ([64] * 16, 4096, 64), ([2000, 0, 1, 17], 1024, 64),
    ([0, 700] + [3] * 300, 256, 64),
]


def test_tile_height_at_its_edges():
    for counts, N, rows in CUT:
        t = tiles(sum(counts), N // 256, np.concatenate([[0], np.cumsum(counts)]), 112)
        assert max(r for _, _, r, _ in t) <= rows, (counts, rows)
        seen = np.zeros((sum(counts), N // 256), int)
        for _, row0, r, nt in t:
            seen[row0:row0 + r, nt] += 1
        assert (seen == 1).all()
        assert rows == 64 or max(r for _, _, r, _ in t) > 64


def small_cols(form, swiglu, E, R, N, K):
    """Columns per workgroup of the small-row kernel, 0: the 256-row one."""
    return _C.lib().smoe_grouped_gemm_small_cols({"plain": 0, "packed": 1, "e8m0": 2}[form], swiglu, E, R, N, K)


@pytest.mark.parametrize("form,swiglu,E,N,K,line", [
    ("plain", True, 16, 2560, 1408, 56),     # 160 tiles of 256 x 256: up to three quarters of a round
    ("plain", False, 24, 2560, 4480, 48),    # 240
    ("plain", True, 32, 2048, 7168, 48),     # 256: a whole round
    ("packed", False, 24, 2560, 7168, 64), ("e8m0", True, 16, 2560, 4480, 64),
    ("plain", True, 8, 4096, 1024, 80),      # 128: half a round
    ("plain", False, 32, 4096, 7168, 40),    # 512: one and a half to two rounds
    ("plain", True, 26, 4096, 2176, 40),     # 416
    ("plain", True, 32, 4096, 2048, 80), ("plain", False, 24, 4096, 7168, 80), ("plain", True, 33, 4096, 7168, 80),
    ("packed", False, 32, 4096, 7168, 112), ("packed", False, 24, 2560, 2048, 112),
    ("e8m0", False, 32, 5760, 2944, 112),
])
def test_lines_between_the_kernels(form, swiglu, E, N, K, line):
    """Few rows per expert under skewed loads lost to the 256-row kernels where
    those have nearly one or two rounds of tiles: the lines are lower there."""
    assert small_cols(form, swiglu, E, E * line, N, K) > 0
    assert small_cols(form, swiglu, E, E * line + 1, N, K) == 0


@pytest.mark.parametrize("E,N,rows,cols", [
    (24, 2560, 8, 64), (24, 2560, 9, 256), (24, 2560, 64, 256), (24, 2560, 65, 128),
    (16, 2560, 16, 64), (16, 2560, 17, 256), (32, 2048, 40, 128), (8, 4096, 40, 64), (128, 2048, 40, 256),
])
def test_columns_per_workgroup(E, N, rows, cols):
    assert small_cols("packed", False, E, E * rows, N, 2048) == cols


# ------------------------------------------------------------------- GPU
def bits(t):
    return t.contiguous().view(torch.uint8 if t.element_size() == 1 else torch.int16
                               if t.element_size() == 2 else torch.int32)


CASES = [
    # counts, N, K: tile and block edges; K of 1, 3 and 5 steps, past 64 and 128 steps
    ([1, 15, 16, 17, 0, 31, 32, 33, 48, 49, 63, 64, 65], 512, 512),
    ([95, 96, 97, 0, 2, 111, 0, 0, 112, 113, 1, 0, 0, 0, 0, 0], 256, 1024),
    ([127, 128, 129, 0, 224, 225, 256, 257, 3, 0, 0, 0, 0, 0], 256, 2048),
    ([1500, 0, 700], 256, 1024),  # few tiles and a short K: many rows per expert
    ([5, 0, 20, 70], 272, 128),
    ([40, 3], 1040, 640),
    ([2, 0, 90, 33], 256, 66 * 128),
    ([33, 7, 0, 60], 256, 132 * 128),
    ([1], 128, 384),
    ([3, 0, 1, 100, 0, 17] * 60, 256, 512),
]


def run(xq, xs, w, ws, off, R, e8m0, swiglu, N):
    """The valid rows' outputs with buffers of R rows; none past offsets[E]
    is written."""
    n = int(off[-1])
    rows = xq.new_empty((R,) + xq.shape[1:])
    sc = xs.new_empty((R,) + xs.shape[1:])
    rows.view(torch.uint8).zero_()
    sc.fill_(1.0)
    rows.view(torch.uint8)[:n], sc[:n] = xq.view(torch.uint8)[:n], xs[:n]
    if swiglu:
        out = ops.grouped_gemm_fp8_swiglu(rows, sc, w, ws, off, save_c1=True, scale="pow2" if e8m0 else "amax")
        return [bits(o[:n]) for o in out]
    out = torch.full((R, N), 7.0, dtype=torch.bfloat16, device=xq.device)
    ops.grouped_gemm_fp8(rows, sc, w, ws, off, out=out, e8m0=e8m0)
    assert (out[n:].float() == 7.0).all()
    return [bits(out[:n])]


@pytest.mark.gpu
@pytest.mark.parametrize("counts,N,K", CASES)
@pytest.mark.parametrize("form", ["plain", "packed", "e8m0"])
def test_small_rows_equal_the_256_row_kernels(dev, counts, N, K, form):
    print("[small]", form, len(counts), N, K, flush=True)
    E, n = len(counts), int(sum(counts))
    e8m0 = form == "e8m0"
    if form != "plain" and not (ops.packed_e8m0_ok if e8m0 else ops.packed_gemm_ok)(N, K):
        with pytest.raises(ValueError):  # refused as before
            wq = torch.zeros((E, N, K), dtype=torch.uint8, device=dev)
            ops.grouped_gemm_fp8(torch.zeros((n, K), dtype=torch.uint8, device=dev),
                                 torch.ones((n, K // 128), device=dev), ops.PackedWeight(wq),
                                 torch.ones((E, -(-N // 128), K // 128), device=dev),
                                 W.offsets_from_counts(counts, dev), e8m0=e8m0)
        return
    scale = "pow2" if e8m0 else "amax"
    off = W.offsets_from_counts(counts, dev)
    x = W.tokens(n, K, device=dev, seed=K + N)
    xq, xs = ops.quant_rows(x, scale=scale)
    wq, ws = ops.quantize_weight_blockwise(W.weights(E, N, K, device=dev, seed=N), scale=scale)
    w = wq if form == "plain" else ops.pack_weight_fp8(wq)
    for swiglu in (False, True):
        if swiglu and N % 256:
            continue
        # over the lines (1024 rows, 96 tiles; short K with SwiGLU 8192 rows): the 256-row kernels
        big = n + max(1025 * E, 97 * 256) + (8192 * E if swiglu and K <= 2048 else 0)
        few = run(xq, xs, w, ws, off, n, e8m0, swiglu, N)
        for a, b in zip(few, run(xq, xs, w, ws, off, big, e8m0, swiglu, N)):
            assert torch.equal(a, b), f"swiglu={swiglu}"
        if not swiglu and K <= 1024 and E < 20:
            ref = O.grouped_gemm_fp8(xq.view(torch.uint8).cpu().numpy(), xs.cpu().numpy(),
                                     wq.view(torch.uint8).cpu().numpy(), ws.cpu().numpy(), off.cpu().numpy())
            got = few[0].view(torch.bfloat16).float().cpu().numpy()
            # bf16 rounds to 2^-9 of a value, about 1.4e-3 on average
            d = np.abs(got - ref)
            assert d.max() <= 1e-2 * np.abs(ref).max() and d.mean() <= 2e-3 * np.abs(ref).mean()


CUT_K = 1536
# (of these only the narrow loads are below the line of plain weights)
CUT_FORMS = [(f, c, N) for c, N, _ in CUT for f in ("plain", "packed", "e8m0") if f != "plain" or N == 256]


@pytest.mark.gpu
@pytest.mark.parametrize("form,counts,N", CUT_FORMS)
def test_tile_heights_equal_the_256_row_kernels(dev, form, counts, N):
    """Both heights of the small-row kernel's tiles, against the 256-row ones."""
    print("[cut]", form, len(counts), N, flush=True)
    E, n, K, e8m0 = len(counts), sum(counts), CUT_K, form == "e8m0"
    big = n + 8193 * E
    assert small_cols(form, True, E, big, N, K) == 0
    assert small_cols(form, True, E, n, N, K) == 256
    scale = "pow2" if e8m0 else "amax"
    off = W.offsets_from_counts(counts, dev)
    xq, xs = ops.quant_rows(W.tokens(n, K, device=dev, seed=n), scale=scale)
    wq, ws = ops.quantize_weight_blockwise(W.weights(E, N, K, device=dev, seed=N), scale=scale)
    w = wq if form == "plain" else ops.pack_weight_fp8(wq)
    for a, b in zip(run(xq, xs, w, ws, off, n, e8m0, True, N), run(xq, xs, w, ws, off, big, e8m0, True, N)):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [3200, 3584])
@pytest.mark.parametrize("form", ["plain", "e8m0"])
def test_short_tiles_of_the_256_row_kernels(dev, K, form):
    """Last tiles on both sides of the 64 and 128 rows at which the 256-row
    kernels (without SwiGLU) skip row blocks, against the same rows in a call
    whose average (above 2048 rows, the rest unused) selects those without the
    skip."""
    print("[short tiles]", form, K, flush=True)
    E, N, e8m0 = 96, 512, form == "e8m0"
    edges = [1, 16, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 385, 449, 512, 700, 0, 900, 1025,
             0, 300]
    counts = edges * 4
    scale = "pow2" if e8m0 else "amax"
    off = W.offsets_from_counts(counts, dev)
    n = sum(counts)
    assert 256 * E <= n <= 1024 * E and (n // 256 + E // 2) * 2 >= 256
    xq, xs = ops.quant_rows(W.tokens(n, K, device=dev, seed=K), scale=scale)
    wq, ws = ops.quantize_weight_blockwise(W.weights(E, N, K, device=dev, seed=3), scale=scale)
    w = ops.pack_weight_fp8(wq) if e8m0 else wq
    short = run(xq, xs, w, ws, off, n, e8m0, False, N)
    for a, b in zip(short, run(xq, xs, w, ws, off, 2049 * E + n, e8m0, False, N)):
        assert torch.equal(a, b)
