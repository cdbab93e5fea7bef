"""The edges of the 256-row grouped GEMMs (smoe_gemm.hip, smoe_gemm_packed.hip,
smoe_gemm_e8m0.hip) and of the small-row kernel, each on its own side of the
lines between them.  A call of few rows takes the small-row kernel; the same
operands with unused rows past offsets[E] take the 256-row one.  The two must
give the same bytes and both are held to the float64 oracle; the CPU part pins
which kernel each shape takes, so that a moved line cannot take a case off the
kernel it is for."""
import sys

import numpy as np
import pytest
import torch

from oracle import smoe_oracle as O
from smoe import _C, ops
from smoe import workloads as W

LAYOUT = {"plain": 0, "packed": 1, "e8m0": 2}
MAX_REL, MEAN_REL = 1e-2, 1e-3  # GEMM outputs against the oracle rounded to bf16


def say(*a):
    print("[edge]", *a, flush=True)
    sys.stdout.flush()


def small_cols(form, swiglu, E, R, N, K):
    """Columns per workgroup of the small-row kernel, 0: the 256-row one."""
    return _C.lib().smoe_grouped_gemm_small_cols(LAYOUT[form], swiglu, E, R, N, K)


def rows_over_the_line(form, swiglu, E, n, N, K):
    """Rows of a buffer that sends n used rows to the 256-row kernel."""
    R = n
    while small_cols(form, swiglu, E, R, N, K):
        R = R * 5 // 4 + 64
    return R


SKEW = [300, 0, 513, 1]
EDGES = [
    # counts, N, K, forms: partial last column tiles (N % 256 of 128, 16, 64 and a lone half tile)
    (SKEW, 384, 512, ("plain", "packed", "e8m0")),
    (SKEW, 784, 1024, ("plain", "packed", "e8m0")),
    (SKEW, 2880, 512, ("plain", "packed", "e8m0")),
    ([100, 200], 128, 512, ("plain", "packed", "e8m0")),
    ([17, 600], 2048, 7168, ("plain", "packed", "e8m0")),
    ([1], 16, 1024, ("plain", "packed", "e8m0")),
    # K blocks in every class of 4 (the E8M0 scale windows end at K), few and many
    ([5, 0, 300, 1, 0, 129, 128, 17], 256, 128, ("plain",)),
    (SKEW, 512, 384, ("plain",)),
    (SKEW, 256, 640, ("plain", "e8m0")), (SKEW, 512, 768, ("plain", "e8m0")),
    (SKEW, 256, 896, ("plain", "e8m0")), ([129, 400], 384, 1152, ("plain", "e8m0")),
    ([600, 77], 2880, 2944, ("plain", "e8m0")),
    # 512 K blocks, the most: the weight scales' table in LDS at its largest
    ([3, 130], 256, 65536, ("plain", "packed", "e8m0")),
    # 1024 experts, the most: several experts per thread of the tile search
    ([0, 7, 39] * 341 + [300], 256, 1024, ("plain", "packed", "e8m0")),
]
EDGES = [(f, c, N, K) for c, N, K, forms in EDGES for f in forms]
ids = [f"{f}-{len(c)}x{sum(c)}-{N}-{K}" for f, c, N, K in EDGES]

SWIGLU = [(f, c, 2 * I, K) for f, c, I, K in [
    ("plain", [20, 0, 77], 256, 1024), ("packed", [200, 0, 333], 256, 1024), ("e8m0", [200, 0, 333], 256, 1024),
    ("packed", [513, 64], 768, 2048), ("e8m0", [257, 3], 384, 640), ("e8m0", [129, 0, 400], 256, 2944),
    ("plain", [1, 60], 128, 640), ("packed", [300, 0, 77], 128, 512)]]


@pytest.mark.parametrize("form,counts,N,K", EDGES, ids=ids)
def test_edges_reach_both_kernels(form, counts, N, K):
    E, n = len(counts), sum(counts)
    assert small_cols(form, False, E, n, N, K) > 0
    R = rows_over_the_line(form, False, E, n, N, K)
    assert n < R and R * K < 4 << 30 and R * N < 1 << 30  # what the GPU part allocates


@pytest.mark.parametrize("form,counts,N,K", SWIGLU)
def test_swiglu_edges_reach_both_kernels(form, counts, N, K):
    E, n = len(counts), sum(counts)
    assert small_cols(form, True, E, n, N, K) == 256
    assert n < rows_over_the_line(form, True, E, n, N, K) <= 2 * 8193 * E + 64


# column tiles of the small-row kernel without SwiGLU: 256, 128 and 64 columns,
# the last one partial, tiles on the edges of the 96, 112 and 128-row loops
TALL = [96, 97, 112, 113, 128, 129, 0, 1, 15, 33, 64, 65, 0, 225, 80, 48]
COLUMNS = [
    # counts, N, columns per workgroup
    (TALL * 2, 5760, 256), ([4 * c // 5 for c in TALL] * 8, 1040, 256),
    (TALL * 2, 2880, 128), ([65] * 16, 2576, 128),
    (TALL * 2, 272, 64), (TALL, 720, 64),
]
# (65 rows are above the line of plain weights)
COLUMNS = [(f, c, N, K, w) for c, N, w in COLUMNS for f, K in [("plain", 512), ("packed", 512), ("e8m0", 640)]
           if f != "plain" or N != 2576]


def test_column_cases_cover_every_width_and_form():
    seen = set()
    for form, counts, N, K, width in COLUMNS:
        assert small_cols(form, False, len(counts), sum(counts), N, K) == width, (form, N)
        assert N % width
        seen.add((form, width))
    assert seen >= {(f, w) for f in LAYOUT for w in (256, 128, 64)}


# ------------------------------------------------------------------- GPU
def u8(t):
    return t.detach().cpu().contiguous().view(torch.uint8).numpy()


def u16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def operands(dev, form, counts, N, K, seed):
    scale = "pow2" if form == "e8m0" else "amax"
    xq, xs = ops.quant_rows(W.tokens(max(sum(counts), 1), K, device=dev, seed=seed), scale=scale)
    wq, ws = ops.quantize_weight_blockwise(W.weights(len(counts), N, K, device=dev, seed=seed + 1), scale=scale)
    return xq, xs, wq, ws, wq if form == "plain" else ops.pack_weight_fp8(wq)


def padded(t, R, fill=0):
    """t with R rows, the new ones unused."""
    out = torch.full((R,) + t.shape[1:], fill, dtype=torch.uint8 if t.element_size() == 1 else t.dtype, device=t.device)
    out[:t.shape[0]] = t.view(out.dtype)
    return out


def gemm(form, xq, xs, w, ws, off, N):
    """[R, N] between guard rows that must keep their value."""
    R = xq.shape[0]
    buf = torch.full((R + 128, N), 7.0, dtype=torch.bfloat16, device=xq.device)
    ops.grouped_gemm_fp8(xq, xs, w, ws, off, out=buf[64:R + 64], e8m0=form == "e8m0")
    assert bool((buf[:64] == 7.0).all()) and bool((buf[R + 64:] == 7.0).all())
    return buf[64:R + 64]


def check_oracle(got, xq, xs, wq, ws, off, rows, what):
    """got's rows against the oracle; off: the offsets, each row in one expert."""
    off = np.asarray(off)
    owner = np.searchsorted(off, rows, side="right") - 1
    soff = np.concatenate([[0], np.cumsum(np.bincount(owner, minlength=off.size - 1))])
    at = torch.from_numpy(rows).to(xq.device)
    ref = O.grouped_gemm_fp8(u8(xq.view(torch.uint8)[at]), xs[at].cpu().numpy(), u8(wq), ws.cpu().numpy(), soff)
    ref = O.bf16_to_f32(O.f32_to_bf16(ref.astype(np.float32))).astype(np.float64)
    d = np.abs(O.bf16_to_f32(u16(got[at])) - ref)
    mx, mn = d.max() / np.abs(ref).max(), d.mean() / np.abs(ref).mean()
    assert mx <= MAX_REL and mn <= MEAN_REL, f"{what}: max_rel={mx:.3e} mean_rel={mn:.3e}"


def some_rows(counts, most=8):
    """Up to `most` rows of every expert, its first and last among them."""
    off = np.concatenate([[0], np.cumsum(counts)])
    return np.unique(np.concatenate([np.linspace(off[e], off[e + 1] - 1, min(most, c)).astype(np.int64)
                                     for e, c in enumerate(counts) if c]))


@pytest.mark.gpu
@pytest.mark.parametrize("form,counts,N,K", EDGES, ids=ids)
def test_edges_of_the_gemms(dev, form, counts, N, K):
    say(form, len(counts), sum(counts), N, K)
    E, n = len(counts), sum(counts)
    R = rows_over_the_line(form, False, E, n, N, K)
    off = W.offsets_from_counts(counts, dev)
    xq, xs, wq, ws, w = operands(dev, form, counts, N, K, N + K)
    few = gemm(form, xq, xs, w, ws, off, N)
    big = gemm(form, padded(xq, R), padded(xs, R, 1.0), w, ws, off, N)
    assert bool((big[n:] == 7.0).all())
    assert torch.equal(few.view(torch.int16), big[:n].view(torch.int16))
    if E > 64:  # the oracle decodes every expert's weights: the first and the last of them
        counts = counts[:8] + [0] * (E - 16) + counts[-8:]
        lead = W.offsets_from_counts([0, 7, 39] * 341 + [300])
        at = np.concatenate([np.arange(int(lead[8])), np.arange(int(lead[-9]), n)])
        sub = torch.from_numpy(at).to(dev)
        xq, xs, big = xq.view(torch.uint8)[sub], xs[sub], big[sub]
    check_oracle(big, xq, xs, wq, ws, np.concatenate([[0], np.cumsum(counts)]), some_rows(counts), "256-row")


@pytest.mark.gpu
@pytest.mark.parametrize("form,counts,N,K", SWIGLU)
def test_swiglu_edges_of_the_gemms(dev, form, counts, N, K):
    say("swiglu", form, counts, N, K)
    E, n, I = len(counts), sum(counts), N // 2
    R = rows_over_the_line(form, True, E, n, N, K)
    off = W.offsets_from_counts(counts, dev)
    xq, xs, wq, ws, w = operands(dev, form, counts, N, K, N + K)
    pow2 = form == "e8m0"
    scale = "pow2" if pow2 else "amax"
    hq, hs, c1 = ops.grouped_gemm_fp8_swiglu(xq, xs, w, ws, off, save_c1=True, scale=scale)
    bhq, bhs, bc1 = ops.grouped_gemm_fp8_swiglu(padded(xq, R), padded(xs, R, 1.0), w, ws, off, save_c1=True, scale=scale)
    assert torch.equal(c1.view(torch.int16), bc1[:n].view(torch.int16))
    assert torch.equal(hq.view(torch.uint8), bhq[:n].view(torch.uint8)) and torch.equal(hs, bhs[:n])
    oq, os_ = O.swiglu_quant(u16(bc1[:n]), pow2=pow2)
    assert np.array_equal(u8(bhq[:n]), oq) and np.array_equal(bhs[:n].cpu().numpy(), os_)
    check_oracle(bc1, xq, xs, wq, ws, np.concatenate([[0], np.cumsum(counts)]), some_rows(counts), "256-row c1")


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "packed", "e8m0"])
def test_row_window_of_the_256_row_kernels(dev, form):
    """offsets that start past row 0: only [offsets[0], offsets[E]) is written."""
    say("row window", form)
    counts, N, K = [40, 260, 0, 255, 45], 512, 1024
    R = rows_over_the_line(form, False, 3, 600, N, K)
    xq, xs, wq, ws, w = operands(dev, form, counts, N, K, 7)
    wq, ws = wq[1:4].contiguous(), ws[1:4].contiguous()
    w = wq if form == "plain" else ops.pack_weight_fp8(wq)
    off = torch.tensor([40, 300, 300, 555], dtype=torch.int32, device=dev)
    got = gemm(form, padded(xq, R), padded(xs, R, 1.0), w, ws, off, N)
    assert bool((got[:40] == 7.0).all()) and bool((got[555:] == 7.0).all())
    check_oracle(got, xq, xs, wq, ws, [40, 300, 300, 555], np.arange(40, 555, 7), form)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "packed", "e8m0"])
def test_malformed_offsets_of_the_256_row_kernels(dev, form):
    """offsets[] is device data that the host does not check, so the kernel
    clamps every tile to rows [0, R): expert 1's offsets decrease (no tiles)
    and expert 2's run past R.  Nothing outside the output is written and the
    rows of one expert alone match the oracle."""
    say("malformed offsets", form)
    N, K = 256, 512
    R = rows_over_the_line(form, False, 3, 1000, N, K)
    xq, xs, wq, ws, w = operands(dev, form, [0, 0, R], N, K, 77)
    off = torch.tensor([0, 400, 300, R + 500], dtype=torch.int32, device=dev)
    got = gemm(form, xq, xs, w, ws, off, N)
    check_oracle(got, xq, xs, wq, ws, [0, 300, 300, 300], np.arange(300), "expert 0")
    rows = np.concatenate([np.arange(400, R, 97), np.arange(R - 300, R)])
    check_oracle(got, xq, xs, wq, ws, [0, 0, 0, R], np.unique(rows), "expert 2, clamped at R")


@pytest.mark.gpu
@pytest.mark.parametrize("form,counts,N,K,width", COLUMNS)
def test_column_tiles_equal_the_256_row_kernels(dev, form, counts, N, K, width):
    say("columns", form, len(counts), N, K, width)
    n = sum(counts)
    R = rows_over_the_line(form, False, len(counts), n, N, K)
    off = W.offsets_from_counts(counts, dev)
    xq, xs, wq, ws, w = operands(dev, form, counts, N, K, N)
    few = gemm(form, xq, xs, w, ws, off, N)
    big = gemm(form, padded(xq, R), padded(xs, R, 1.0), w, ws, off, N)
    assert torch.equal(few.view(torch.int16), big[:n].view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(8))
def test_random_shapes_on_both_kernels(dev, seed):
    rng = np.random.default_rng(200 + seed)
    E = int(rng.integers(1, 24))
    counts = np.where(rng.random(E) < 0.2, 0, rng.integers(1, 200, E)).tolist()
    counts[0] += 1
    N, K = 16 * int(rng.integers(1, 65)), 128 * int(rng.choice([1, 2, 3, 4, 5, 6, 8, 12, 16]))
    say("random", seed, counts, N, K)
    n, off = sum(counts), W.offsets_from_counts(counts, dev)
    for form in LAYOUT:
        if form != "plain" and not (ops.packed_gemm_ok if form == "packed" else ops.packed_e8m0_ok)(N, K):
            continue
        R = rows_over_the_line(form, False, E, n, N, K)
        xq, xs, wq, ws, w = operands(dev, form, counts, N, K, 300 + seed)
        few = gemm(form, xq, xs, w, ws, off, N)
        big = gemm(form, padded(xq, R), padded(xs, R, 1.0), w, ws, off, N)
        assert torch.equal(few.view(torch.int16), big[:n].view(torch.int16))
        check_oracle(big, xq, xs, wq, ws, off.cpu().numpy(), some_rows(counts), f"{form} seed {seed}")
