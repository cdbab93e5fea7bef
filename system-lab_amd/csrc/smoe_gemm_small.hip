// smoe_gemm_small.hip — the dropless fp8 grouped GEMM for few rows per expert
// (decode batches, short prompt chunks), for gfx950.
//
//   c[r,n] = bf16( sum_kb as[r,kb] * bs[e,n/128,kb] * sum_{k in kb} a[r,k]*b[e,n,k] )
//
// Contract, K orders and arithmetic per output are those of the 256-row
// kernels (smoe_gemm.hip for plain weights, smoe_gemm_packed.hip for packed
// ones, smoe_gemm_e8m0.hip for power-of-two scales), so the bytes are the
// same.  What differs is the shape of the problem: with a few dozen rows per
// expert every weight byte is used by one tile or two, and the time is that
// of streaming the weights of the experts that have rows from HBM.
//
// Tiling.  A workgroup of 4 waves owns up to 112 rows (128 with E8M0 scales,
// which need no registers for the MFMA's products) x 64*kCB columns; wave w
// owns all rows and columns w*16*kCB .. +16*kCB.  The weights go straight
// from memory to the MFMA operand registers (nothing else in the workgroup
// needs them), kD K steps ahead.  The row count of a tile picks its loop: 1,
// 2, 4, 6 or 7 (8) blocks of 16 rows, so a tile of one row does a sixteenth of
// a 256-row tile's MFMAs.  The activations of a tile pass through LDS in chunks
// of at most 16 KiB (8, 4, 2 or 1 K steps), loaded to registers a chunk ahead
// and written to the other half of the buffer at the chunk's end: one barrier
// a chunk.  All loads are ordinary ones, so the compiler counts and waits for
// each.  At most 256 registers and 68 KiB of LDS leave two workgroups per
// CU, so one tile's start and end hide behind the other's stream.
//
// With 65 rows or more and few tiles the workgroup may take 64 rows instead
// (find_tile decides, see kLowRows).
//
// Every wave finds the workgroup's tile by itself (wave scans over the
// experts' tile counts): no LDS and no barrier before the first load.
// Tiles are numbered expert by expert and dealt to the XCDs in 8 contiguous
// ranges; within an expert the row tiles of one column tile are neighbours,
// so they share the weights in one L2 (with the column tiles fastest, 100
// rows an expert at N = 28672, K = 4096 took 294 us against 237).
//
// Measured against the 256-row kernels (router loads, us before -> after):
// H 4096, I 14336, E 8, 32 tokens top-2: fc1 with SwiGLU 261 -> 160 (5.9 TB/s
// of weights), fc2 162 -> 81 (5.8 TB/s); H 2048, I 768, E 128, top-8: fc1 with
// SwiGLU 29 -> 20 at 1 token, 122 -> 70 at 64 (5.8 TB/s), 125 -> 97 at 1000;
// its fc2 on plain weights 65 -> 40 at 64 tokens, with E8M0 scales 72 -> 33.
// Tiles of up to 96 rows instead of 112 / 128: H = I = 2880, E 32, 777 tokens top-4
// (97 rows) E8M0 fc1 151 -> 135, fc2 80 -> 62.  Loading the 64-row loop's weights
// three steps ahead instead of two changed nothing but a 37-row case (5% slower).
#include "smoe_gemm_small.h"
#include "smoe_mfma.h"

namespace smoe {
namespace small {

constexpr int kThreads = 256, kWaves = 4;
// Most rows of a tile: what the registers hold beside two K steps of weights
// (128 accumulators a lane, which spills two registers, or 112 and the
// products the scales multiply).
template <bool kE8>
constexpr int kTileRows = kE8 ? 128 : 112;
constexpr int kMaxChunk = 16 * 1024;  // most activation bytes of a chunk

// Tall experts are cut into tiles of kLowRows rows instead of kTileRows while
// the launch then still has at most two workgroups per CU (kLowMax): its time
// is that of its tallest tile, a taller loop waits longer per K step (the 64-row
// loop takes two K steps of activations at once), and the experts' sizes
// are only known here.  Not where the tall tiles would have a CU each and the
// low ones not (kCUs): a CU with two tiles streams twice the weights.  us without ->
// with (fused SwiGLU; the 256-row kernels in brackets), Zipf(1.2) loads: E 128, N
// 1536, K 2048, 128 rows, packed 29.1 -> 18.8 (32.3); E 96, N 1024, K 4608, 192 rows, plain
// 68.6 -> 42.9 (64.0); E 16, N 4608, K 3584, 512 rows, packed 79.7 -> 61.1 (83.0);
// random loads: E 8, N 4096, K 1024, 512 rows, plain 26.2 -> 18.9 (23.0).
constexpr int kLowRows = 64, kLowMax = 512, kCUs = 256;

struct Tile {
  int row0, rows, e, nt;
};

// The tile of workgroup bid: false when it is past the last one.  offsets[] is
// device data the host never sees: whatever it holds, rows stay in [0, R).
// low: the height of the tiles is chosen here.  An expert's rows are then at
// most R <= kLowMax * kLowRows, so counts of both heights share a word (64
// experts' sums stay below 2^16) and need no bound of their own.
template <int kBM>
__device__ __forceinline__ bool find_tile(const int32_t* __restrict__ offsets, int E, int R, int NT,
                                          int mt_bound, bool low, int bid, int lane, Tile& t) {
  auto row_at = [&](int e) { return max(0, min(offsets[min(e, E)], R)); };
  // tiles of an expert; with low, those of kLowRows rows in the high half
  auto tiles = [&](int e) {
    const int n = max(row_at(e + 1) - row_at(e), 0);
    const int c = min((n + kBM - 1) / kBM, mt_bound);
    return low ? c | (n + kLowRows - 1) / kLowRows << 16 : c;
  };
  auto scan = [&](int v) {
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int u = __shfl_up(v, o, kWave);
      if (lane >= o) v += u;
    }
    return v;
  };
  constexpr int kHeld = 4;  // experts a lane keeps between the two passes
  int cnt[kHeld], inc[kHeld];
#pragma unroll
  for (int i = 0; i < kHeld; ++i) cnt[i] = tiles(i * kWave + lane);
  int total = 0, total_low = 0;
  auto add = [&](int v) {
    total = min(total + (low ? v & 0xffff : v), mt_bound);
    total_low += (int)((uint32_t)v >> 16);
  };
#pragma unroll
  for (int i = 0; i < kHeld; ++i) {
    if (i * kWave < E) {
      inc[i] = scan(cnt[i]);
      add(__builtin_amdgcn_readlane(inc[i], kWave - 1));
    }
  }
  for (int b = kHeld * kWave; b < E; b += kWave)
    add(__builtin_amdgcn_readlane(scan(tiles(b + lane)), kWave - 1));
  const bool cut = low && total_low * NT <= kLowMax && !(total * NT <= kCUs && total_low * NT > kCUs);
  const int bm = cut ? kLowRows : kBM;
  if (cut) total = total_low;
  auto count = [&](int v) { return low ? (cut ? (int)((uint32_t)v >> 16) : v & 0xffff) : v; };
  // 8 contiguous ranges of tiles, one per XCD; an expert's row tiles of one
  // column tile are neighbours, so its weights are read from memory once
  const int all = total * NT;
  const int chunk = (all + 7) / 8;
  const int j = bid >> 3, tl = (bid & 7) * chunk + j;
  if (j >= chunk || tl >= all) return false;
  const int mt = tl / NT;  // a row tile of the expert
  int carry = 0, nt_e = 1, first = 0;
  auto take = [&](int b, int c, int v) {  // the 64 experts from b: counts c, inclusive scan v
    const uint64_t past = __ballot(carry + v > mt);
    if (!past) {
      carry += __builtin_amdgcn_readlane(v, kWave - 1);
      return false;
    }
    const int l = __builtin_ctzll(past);
    t.e = b + l;
    nt_e = __builtin_amdgcn_readlane(c, l);
    first = carry + __builtin_amdgcn_readlane(v, l) - nt_e;
    return true;
  };
  bool found = false;
#pragma unroll
  for (int i = 0; i < kHeld; ++i)
    if (!found && i * kWave < E) found = take(i * kWave, count(cnt[i]), count(inc[i]));
  for (int b = kHeld * kWave; b < E && !found; b += kWave) {
    const int c = count(tiles(b + lane));
    found = take(b, c, scan(c));
  }
  if (!found || t.e >= E) return false;
  const int q = tl - first * NT;
  t.nt = q / nt_e;
  // the expert's n rows in nt_e = ceil(n / bm) tiles of equal height, a
  // multiple of 16: at most bm, so the last one is never empty
  const int o0 = row_at(t.e), o1 = row_at(t.e + 1);
  const int h = min(((o1 - o0 + nt_e - 1) / nt_e + 15) & ~15, bm);
  t.row0 = o0 + (q - t.nt * nt_e) * h;
  t.rows = min(h, o1 - t.row0);
  return t.rows > 0;
}

__device__ __forceinline__ int e8m0_of(float s) { return (__float_as_uint(s) >> 23) & 0xff; }

__device__ __forceinline__ v8i lds_frag2(const uint8_t* base, int row, int c0, int c1) {
  const v4i lo = *(const v4i*)(base + swz(row, c0));
  const v4i hi = *(const v4i*)(base + swz(row, c1));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// The K loop of a tile of at most 16*kRB rows and its bf16 result staged in
// LDS (row pitch kCPitch).  kD: K steps the weights are loaded ahead.
template <SmallWeights kLay, bool kE8, int kCB, int kRB, int kD>
__device__ __forceinline__ void run_tile(const uint8_t* __restrict__ a_base,
                                         const float* __restrict__ s_base,
                                         const uint8_t* __restrict__ b_base,
                                         const float* __restrict__ sb_row, const uint32_t (&ob)[kCB],
                                         int rows, int Kd, int ksb, uint8_t* smem, int tid) {
  constexpr int kS = kRB <= 2 ? 8 / kRB : kRB == 4 ? 2 : 1;  // K steps per chunk
  constexpr int kLB = kRB == 7 ? 8 : kRB;  // row blocks loaded: whole segments for every wave
  constexpr int kStep = kLB * 16 * kRow;  // LDS bytes per step
  constexpr int kChunk = kS * kStep, kQ = kChunk / (kThreads * 16);
  constexpr int kWords = kS * kLB * 16;  // activation scales of a chunk
  constexpr bool kPacked = kLay == SmallWeights::kPacked;
  constexpr int kHalf = kPacked ? 1024 : 16;     // a weight fragment's second 16 bytes
  constexpr int kKStep = kPacked ? 2048 : kBK;   // weight bytes from one K block to the next
  constexpr int kCPitch = 64 * kCB * 2 + 16;
  static_assert(kQ * kThreads * 16 == kChunk && kChunk <= kMaxChunk && kWords <= kThreads, "chunk");
  const int lane = tid & 63, wid = tid >> 6;
  const int frow = lane & 15, fg = lane >> 4;

  // this thread's 16-byte pieces of a chunk: 1 KiB segment q*4 + wid
  // holds 8 row positions of one step (layout as in smoe_mfma.h)
  uint32_t oa[kQ];
  int sa[kQ];
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    const int seg = q * kWaves + wid;
    const int st = seg / (kLB * 2), rg = seg % (kLB * 2);
    const int row = tile_row(rg * 8 + (lane >> 3));
    oa[q] = (uint32_t)(min(row, rows - 1) * Kd + (((lane & 7) ^ (row & 7)) << 4));
    sa[q] = st;
  }
  // threads below kWords also carry one activation scale
  const int s_row = tid % (kLB * 16), s_st = (tid / (kLB * 16)) % kS;
  const uint32_t os = (uint32_t)(min(s_row, rows - 1) * ksb);
  v4i stg[kQ];
  float sstg;
  auto fetch = [&](int kc) {  // the chunk from K step kc (steps past the end repeat the last)
#pragma unroll
    for (int q = 0; q < kQ; ++q)
      stg[q] = *(const v4i*)(a_base + oa[q] + (size_t)min(kc + sa[q], ksb - 1) * kBK);
    sstg = s_base[os + min(kc + s_st, ksb - 1)];
  };
  auto stash = [&](int half) {
    uint8_t* d = smem + half * kChunk + wid * 1024 + lane * 16;
#pragma unroll
    for (int q = 0; q < kQ; ++q) *(v4i*)(d + q * kWaves * 1024) = stg[q];
    if (tid < kWords) ((float*)(smem + 2 * kChunk))[half * kWords + tid] = sstg;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  v8i w[kD][kCB];
  auto load_w = [&](int kb, v8i (&f)[kCB]) {
    const uint8_t* base = b_base + (size_t)kb * kKStep;
#pragma unroll
    for (int j = 0; j < kCB; ++j) {
      const v4i lo = *(const v4i*)(base + ob[j]);
      const v4i hi = *(const v4i*)(base + ob[j] + kHalf);
      f[j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  // activation fragment of 16 tile rows, lane group fg's share of the K block
  // in the weights' order
  auto frag = [&](const uint8_t* sA, int i) {
    const int r = i * 16 + frow;
    return kPacked ? lds_frag2(sA, r, fg, fg + 4) : lds_frag2(sA, r, fg * 2, fg * 2 + 1);
  };
  v4f acc[kRB][kCB];
#pragma unroll
  for (int i = 0; i < kRB; ++i)
#pragma unroll
    for (int j = 0; j < kCB; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

  fetch(0);
#pragma unroll
  for (int d = 0; d < kD; ++d) load_w(min(d, ksb - 1), w[d]);
  // the weight scales of 64 K steps, lane l holding step l of them
  float sbv = sb_row[min(lane, ksb - 1)], sbn = sb_row[min(64 + lane, ksb - 1)];
  stash(0);

  auto step = [&](int kb, v8i (&f)[kCB]) {
    const int half = (kb / kS) & 1;
    const uint8_t* sA = smem + half * kChunk + (kb % kS) * kStep;
    const float* sS = (const float*)(smem + 2 * kChunk) + half * kWords + (kb % kS) * kLB * 16;
    const float sb = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sbv), kb & 63));
    v8i fx = frag(sA, 0);
#pragma unroll
    for (int i = 0; i < kRB; ++i) {
      v8i fxn = fx;
      if (i + 1 < kRB) fxn = frag(sA, i + 1);
      // the empty asm statements keep the row blocks in order (without them
      // the compiler holds the results of a whole step at once)
      asm volatile("" : "+v"(fx));
      if constexpr (kE8) {
        const int ew = e8m0_of(sb), ex = e8m0_of(sS[i * 16 + frow]);
#pragma unroll
        for (int j = 0; j < kCB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(f[j], fx, acc[i][j], 0, 0, 0, ew, 0, ex);
#pragma unroll
        for (int j = 0; j < kCB; ++j) asm volatile("" : "+v"(acc[i][j]));
      } else {
        const float sc = sS[i * 16 + frow] * sb;
        v4f p[kCB];
#pragma unroll
        for (int j = 0; j < kCB; ++j) p[j] = mfma16(f[j], fx, v4f{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
        for (int j = 0; j < kCB; ++j) {
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[i][j][v] = __builtin_fmaf(p[j][v], sc, acc[i][j][v]);
          asm volatile("" : "+v"(acc[i][j]));
        }
      }
      fx = fxn;
    }
    // the buffer just used takes the weights kD steps ahead
    load_w(min(kb + kD, ksb - 1), f);
    asm volatile("" ::: "memory");
  };
  auto at = [&](int kb, v8i (&f)[kCB]) {
    if (kb % kS == 0) fetch(kb + kS);
    step(kb, f);
    if (kb % kS == kS - 1) {
      if ((kb & 63) == 63) {  // kS divides 64
        sbv = sbn;
        sbn = sb_row[min(kb + 65 + lane, ksb - 1)];
      }
      stash(((kb / kS) & 1) ^ 1);
    }
  };
  int kb = 0;
  for (; kb + kD <= ksb; kb += kD) {
#pragma unroll
    for (int d = 0; d < kD; ++d) at(kb + d, w[d]);
  }
#pragma unroll
  for (int d = 0; d < kD - 1; ++d)
    if (kb + d < ksb) at(kb + d, w[d]);

  // ---- bf16 tile over the chunk buffers (every wave is done with them)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int i = 0; i < kRB; ++i)
#pragma unroll
    for (int j = 0; j < kCB; ++j) {
      uint2 o;
      o.x = bf16_pack2(acc[i][j][0], acc[i][j][1]);
      o.y = bf16_pack2(acc[i][j][2], acc[i][j][3]);
      *(uint2*)(smem + (i * 16 + frow) * kCPitch + (wid * 16 * kCB + j * 16 + fg * 4) * 2) = o;
    }
}

template <SmallWeights kLay, bool kE8, bool kSwiGLU, int kCB>
__global__ __launch_bounds__(kThreads, 2) void gemm_small_kernel(
    const uint8_t* __restrict__ a, const float* __restrict__ as, const uint8_t* __restrict__ b,
    const float* __restrict__ bs, const int32_t* __restrict__ offsets, int E, int R, int N, int Kd,
    int mt_bound, bool low, uint16_t* __restrict__ c, uint8_t* __restrict__ hq,
    float* __restrict__ hs) {
  static_assert(!kSwiGLU || kCB == 4, "fused SwiGLU pairs 128 gate with 128 up columns");
  constexpr int kBN = 64 * kCB, kCPitch = kBN * 2 + 16, kBM = kTileRows<kE8>;
  constexpr int kLoop = 2 * kMaxChunk + 2 * kThreads * 4;
  constexpr int kSmem = kLoop > kBM * kCPitch ? kLoop : kBM * kCPitch;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kSmem];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int I = N / 2;
  const int NT = kSwiGLU ? I / kGroup : (N + kBN - 1) / kBN;
  Tile t;
  if (!find_tile<kBM>(offsets, E, R, NT, mt_bound, low, blockIdx.x, lane, t)) return;  // the whole workgroup leaves
  const int e = t.e, row0 = t.row0, rows = t.rows, nt = t.nt;
  const int n0 = nt * kBN, ksb = Kd / kBK, NB = (N + kGroup - 1) / kGroup;

  const uint8_t* a_base = a + (size_t)row0 * Kd;
  const float* s_base = as + (size_t)row0 * ksb;
  // the wave's column blocks (columns past N: clamped, never stored)
  const uint8_t* b_base;
  uint32_t ob[kCB];
  if constexpr (kLay == SmallWeights::kPacked) b_base = b + (size_t)e * ((size_t)N * Kd);
  else b_base = b + ((size_t)e * N + (kSwiGLU ? 0 : n0)) * Kd;
#pragma unroll
  for (int j = 0; j < kCB; ++j) {
    const int wr0 = kSwiGLU ? (wid < 2 ? 0 : I) + nt * kGroup + (wid & 1) * 64 + j * 16
                            : min(n0 + wid * 16 * kCB + j * 16, N - 16);
    if constexpr (kLay == SmallWeights::kPacked)
      ob[j] = (uint32_t)(wr0 / 16) * (uint32_t)ksb * 2048u + (uint32_t)lane * 16u;
    else
      ob[j] = (uint32_t)((wr0 - (kSwiGLU ? 0 : n0) + (lane & 15)) * Kd + (lane >> 4) * 32);
  }
  const int blk = kSwiGLU ? (wid < 2 ? nt : I / kGroup + nt)
                          : min((n0 + wid * 16 * kCB) / kGroup, NB - 1);
  const float* sb_row = bs + ((size_t)e * NB + blk) * ksb;

  if (rows <= 16) run_tile<kLay, kE8, kCB, 1, 4>(a_base, s_base, b_base, sb_row, ob, rows, Kd, ksb, smem, tid);
  else if (rows <= 32) run_tile<kLay, kE8, kCB, 2, 4>(a_base, s_base, b_base, sb_row, ob, rows, Kd, ksb, smem, tid);
  else if (rows <= 64) run_tile<kLay, kE8, kCB, 4, 2>(a_base, s_base, b_base, sb_row, ob, rows, Kd, ksb, smem, tid);
  else if (rows <= 96) run_tile<kLay, kE8, kCB, 6, 2>(a_base, s_base, b_base, sb_row, ob, rows, Kd, ksb, smem, tid);
  else run_tile<kLay, kE8, kCB, kBM / 16, 2>(a_base, s_base, b_base, sb_row, ob, rows, Kd, ksb, smem, tid);
  __syncthreads();

  if constexpr (kSwiGLU) {
    // 8 lanes per row, 16 columns each: h = silu(g) * u from the staged bf16
    // values, amax over the 8 lanes, 16 fp8 bytes per lane
    for (int idx = tid; idx < rows * 8; idx += kThreads) {
      const int r = idx >> 3, sub = idx & 7;
      const uint8_t* rowp = smem + r * kCPitch;
      float fgt[16], fu[16], h[16];
      unpack_bf16x8(*(const uint4*)(rowp + sub * 32), fgt);
      unpack_bf16x8(*(const uint4*)(rowp + sub * 32 + 16), fgt + 8);
      unpack_bf16x8(*(const uint4*)(rowp + 256 + sub * 32), fu);
      unpack_bf16x8(*(const uint4*)(rowp + 256 + sub * 32 + 16), fu + 8);
#pragma unroll
      for (int i = 0; i < 16; ++i) h[i] = silu32(fgt[i]) * fu[i];
      const Q16 q = quant16<kE8>(h);
      const size_t gr = (size_t)(row0 + r);
      *(uint4*)(hq + gr * I + nt * kGroup + sub * 16) = q.q;
      if (sub == 0) hs[gr * (I / kGroup) + nt] = q.scale;
      if (c) {
        uint16_t* crow = c + gr * N + nt * kGroup + sub * 16;
        *(uint4*)crow = *(const uint4*)(rowp + sub * 32);
        *(uint4*)(crow + 8) = *(const uint4*)(rowp + sub * 32 + 16);
        *(uint4*)(crow + I) = *(const uint4*)(rowp + 256 + sub * 32);
        *(uint4*)(crow + I + 8) = *(const uint4*)(rowp + 256 + sub * 32 + 16);
      }
    }
  } else {
    constexpr int kChunks = kBN / 8;  // 16-byte pieces of an output row
    const int ncols = min(kBN, N - n0);
    for (int idx = tid; idx < rows * kChunks; idx += kThreads) {
      const int r = idx / kChunks, ch = idx % kChunks;
      if (ch * 8 < ncols)
        *(uint4*)(c + (size_t)(row0 + r) * N + n0 + ch * 8) = *(const uint4*)(smem + r * kCPitch + ch * 16);
    }
  }
}

}  // namespace small

// The lines between this kernel and the 256-row ones, on the average rows per
// expert (the host knows no more) and the shape.  256-row kernel -> this one in
// us at random loads of the R rows.
//
// 1. One tile per expert: an expert's rows mostly fit one tile and its weights
// are streamed once; past the line the second tile's pass over them costs more
// than the 256-row tile's idle MFMAs.
//   packed, 112 rows: N 1536, K 2048, E 128 150 -> 115; N 28672, K 4096, E 8 272 ->
//     248; N 4096, K 7168, E 32 274 -> 257; at 192 rows 129 -> 148, 279 -> 274, 263 ->
//     328
//   packed E8M0, whose 256-row kernel skips empty row blocks, 112 rows: 111 -> 105,
//     212 -> 198, 204 -> 254 (at 88 rows and Zipf loads 218 -> 235); at 192 rows 126 ->
//     129, 261 -> 262, 239 -> 269
//   N 4096, K 14336, E 8, few and long tiles: 75 rows 163 -> 131, 100 rows 163 -> 190,
//     E8M0 112 rows 132 -> 141, 75 rows and Zipf loads 158 -> 181
//   plain, whose fragment loads touch 16 lines each: 65 rows (N 4096, K 7168) 246 ->
//     199, 97 rows (N 5760, K 2944) 130 -> 152, 100 rows (N 4096, K 7168) 249 -> 289
// Zipf(1.2) loads gain less near the line, where their tall experts' tiles make
// a second, nearly empty round of workgroups: 0.91 - 1.2 of random ones (packed
// 100 rows, N 4096, K 7168: 291 -> 227).  Not so well with plain weights: see 5.
//
// 2. A chip that 256 x 256 tiles leave mostly idle, any rows per expert: up to 96
// such tiles this kernel's more and smaller ones gain 1.04 - 2.7 (E 8, N 1024, 512
// rows: K 2048 30.4 -> 25.6, K 4096 49.1 -> 41.2, plain 32.8 -> 29.1 and 55.5 -> 51.8),
// at 112 0.83 - 1.11, from 144 on 0.63 - 1.07.  Not the plain SwiGLU form (0.91 - 1.36).
//
// 3. A short K in packed form, where a lone 256-row workgroup's prologue and
// epilogue are most of its time and the second workgroup of a CU hides them
// here.  Fused SwiGLU, whose epilogue is the longest:
//   any rows: K <= 1536 1.05 - 1.43, E8M0 K <= 2048 1.02 - 1.9 (N 1536, E 128, 1024
//     rows 1.14; N 768, 128 rows 0.95), both measured to 8192 rows
//   256 - 1024 rows, a second and partly filled 256-row tile: K 2048 1.03 - 1.34
//     (N 1536, E 128, 1024 rows 1.04), E8M0 K 2560 and 3072 1.01 - 1.36; above that
//     0.96 - 1.03 and 0.93 - 1.07, at 192 rows (E8M0 K 2944) 0.92
// and without the epilogue K < 1024: E8M0 to 1024 rows 1.01 - 1.48 (N 2048, K 768,
// E 128: 512 rows 213 -> 195; at 2048 rows and N 256 0.86), K 512 to 512 rows 1.03 -
// 1.53 (at 1024 rows 0.98).
//
// 4. Between half a round and one round of 256 x 256 tiles if every expert has
// one (128 < E * N/256 <= 256) the 256-row kernels stream at their best and this
// one gains least.  45 shapes (E 8 - 64, K 1408 - 7168), means and the
// worst, fused SwiGLU / without, random then Zipf(1.2) loads:
//   plain, up to 192 tiles: 56 rows 1.27 (1.20) / 1.28 (1.24), 1.35 (0.95) / 1.22 (0.91); 72
//     rows 0.87 (0.84) / 80 rows 0.88 (0.84).  Above 192: 48 rows 1.16 (0.88) / 1.19 (0.90),
//     1.05 (0.94) / 0.94 (0.86); 56 rows 0.90 (0.87) / 0.93 (0.89), 1.03 (0.91) / 0.90 (0.85)
//   packed, K > 3072: 64 rows 1.12 (0.92) / 1.13 (0.95), 1.22 (0.98) / 1.16 (0.95); 72 rows
//     0.96 (0.88) with SwiGLU; E8M0 64 rows 1.11 (0.95) / 1.11 (0.96), 72 rows 0.98 (0.95)
//     with SwiGLU.  K <= 3072: as in 1.
//
// 5. Between one and a half and two rounds (384 < E * N/256 <= 512): experts with a
// second tile push the launch past two workgroups per CU, and the few that are
// over run alone.  Means and the worst, with SwiGLU / without, random then
// Zipf(1.2) loads:
//   plain, K > 2048 (13 shapes, E 8 - 96, K 3072 - 14336): 40 rows 1.28 (1.20) / 1.25
//     (1.11), 1.20 (0.99) / 1.09 (0.95); 44 rows 1.26 (1.19) / 1.18 (1.07), 1.05 (0.89) / 1.02
//     (0.84); 48 - 80 rows 1.16 (1.03) / 1.08 (0.87), 0.99 (0.84) / 0.95 (0.79)
//   plain, K 2048, 48 - 80 rows: 1.40 (1.31) / 1.35 (1.18), 1.11 (0.91) / 1.04 (0.92)
//   the packed forms stream faster and keep 1's lines: E8M0 48 - 80 rows 1.32 (1.16) /
//     1.24 (0.96), 1.21 (0.91) / 1.11 (0.89); packed 48 - 88 rows 1.38 (1.22) / 1.31 (1.01),
//     1.20 (0.96) / 1.15 (0.93), 96 - 112 rows 1.09 (0.90) / 1.06 (0.87), 1.28 (1.01) / 1.23 (0.96)
bool small_gemm_rows(SmallWeights lay, bool e8m0, bool swiglu, int E, int R, int N, int Kdim) {
  const bool packed = lay == SmallWeights::kPacked;
  long long one_tile = !packed ? 80
                       : e8m0  ? (Kdim <= 4096 ? 112 : Kdim <= 8192 ? 80 : 64)
                               : (Kdim <= 8192 ? 112 : 80);
  const long long t256 = (N + 255) / 256 * (long long)E;
  if (t256 > 128 && t256 <= 256) {
    if (!packed) one_tile = t256 <= 192 ? 56 : 48;
    else if (Kdim > 3072) one_tile = 64;
  }
  if (!packed && t256 > 384 && t256 <= 512 && Kdim > 2048) one_tile = 40;
  auto to = [&](long long rows) { return R <= rows * E; };
  if (to(one_tile)) return true;
  if ((packed || !swiglu) && (2LL * R + 256LL * E) * ((N + 255) / 256) <= 96 * 512) return true;
  if (!packed) return false;
  if (!swiglu) return Kdim < 1024 && to(e8m0 ? 1024 : 512);
  if (Kdim <= (e8m0 ? 2048 : 1536)) return to(8192);
  return Kdim <= (e8m0 ? 3072 : 2048) && R >= 256LL * E && to(1024);
}

// Column tiles of 64 * small_gemm_cols columns: 4, or without SwiGLU 2 or 1.
// Narrower while the launch has fewer than two workgroups per CU, because few
// workgroups stream too little.  Not so from 16 rows per expert on (8 above
// 192 tiles) where 256 columns make half a round to a round of workgroups, one
// per expert and column tile: narrower ones are then two or four rounds that
// each read the activations again.  45 shapes (as in 4 above), former width -> this
// one, means against the 256-row kernels, random and Zipf(1.2) loads: plain 32 rows
// 1.26 -> 1.33, 1.08 -> 1.25; packed 48 rows 1.24 -> 1.35, 1.03 -> 1.18; E8M0 56 rows 1.13 ->
// 1.23, 1.04 -> 1.17.  Above 64 rows, two tiles an expert, 128 columns: packed 80 rows
// 1.07 -> 1.15, 0.95 -> 1.12.  At fewer rows random loads prefer the narrow ones (up to
// 192 tiles, plain 10 rows 1.51 against 1.41), and at 256 tiles, 512 workgroups of
// 128 columns, they stay ahead (E 32, N 2048, packed 48 rows 1.25 against 1.09).
int small_gemm_cols(bool swiglu, int E, int R, int N) {
  if (swiglu) return 4;
  const long long t256 = (N + 255) / 256 * (long long)E;
  if (t256 > 128 && t256 < 256 && R > (t256 <= 192 ? 16LL : 8LL) * E) return R > (long long)small::kLowRows * E ? 2 : 4;
  const long long live = E < R ? E : R;
  int cb = 4;
  while (cb > 1 && live * (long long)((N + 64 * cb - 1) / (64 * cb)) < 512) cb >>= 1;
  return cb;
}

int small_gemm_launch(SmallWeights lay, bool e8m0, const uint8_t* a, const float* as,
                      const uint8_t* b, const float* bs, const int32_t* offsets, int E, int R,
                      int N, int Kdim, uint16_t* c, uint8_t* hq, float* hs, hipStream_t stream) {
  // at most min(E, R) experts have rows, and each adds at most one partial tile
  // to the R rows' whole ones (the slack serves offsets that overlap)
  const int live = E < R ? E : R;
  const int bm = e8m0 ? small::kTileRows<true> : small::kTileRows<false>;
  const long long mt = live + ((long long)R + bm - 1) / bm;
  const bool swiglu = hq != nullptr;
  const int cb = small_gemm_cols(swiglu, E, R, N);
  const long long NT = swiglu ? N / 2 / kGroup : (N + 64 * cb - 1) / (64 * cb);
  // the kernel may take kLowRows rows per tile where that can fit kLowMax: the
  // grid then holds kLowMax workgroups of them, or all there can be
  const long long cut = ((long long)R + small::kLowRows - 1) / small::kLowRows;
  const bool low = R > small::kLowRows && cut * NT <= small::kLowMax;
  long long bound = mt;
  if (low) {
    const long long fit = (small::kLowMax + NT - 1) / NT;
    bound = live + cut < fit ? live + cut : fit;
    if (bound < mt) bound = mt;
  }
  const long long nblk = (bound * NT + 7) / 8 * 8;
  if (nblk > 0x7fffffffLL) return SMOE_EINVAL_DIM;
#define SMOE_SG(LAY, E8, SW, CB)                                                                \
  small::gemm_small_kernel<SmallWeights::LAY, E8, SW, CB>                                        \
      <<<dim3((unsigned)nblk), dim3(small::kThreads), 0, stream>>>(a, as, b, bs, offsets, E, R, \
                                                                   N, Kdim, (int)bound, low, c, hq, hs)
#define SMOE_SG_CB(LAY, E8)                    \
  do {                                         \
    if (swiglu) SMOE_SG(LAY, E8, true, 4);     \
    else if (cb == 4) SMOE_SG(LAY, E8, false, 4); \
    else if (cb == 2) SMOE_SG(LAY, E8, false, 2); \
    else SMOE_SG(LAY, E8, false, 1);           \
  } while (0)
  if (lay == SmallWeights::kPlain) SMOE_SG_CB(kPlain, false);
  else if (e8m0) SMOE_SG_CB(kPacked, true);
  else SMOE_SG_CB(kPacked, false);
#undef SMOE_SG_CB
#undef SMOE_SG
  SMOE_RETURN_LAUNCH();
}

}  // namespace smoe

extern "C" int smoe_grouped_gemm_small_cols(int layout, int swiglu, int E, int R, int N, int Kdim) {
  using namespace smoe;
  if (E <= 0 || R <= 0 || N <= 0 || Kdim <= 0 || layout < 0 || layout > 2) return 0;
  const SmallWeights lay = layout ? SmallWeights::kPacked : SmallWeights::kPlain;
  if (!small_gemm_rows(lay, layout == 2, swiglu != 0, E, R, N, Kdim)) return 0;
  return 64 * small_gemm_cols(swiglu != 0, E, R, N);
}
