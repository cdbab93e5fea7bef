// smoe_layer.hip — the expert layer's forward and backward as one call each.
//
// A step of the layer is 5 to 20 launches; issued one operator at a time
// from Python, the checks, allocations and calls of those operators took
// longer than the GPU work of a decode step or of a small training step.
// These entry points enqueue the same launches in the same order on the same
// streams from one call, with the intermediates carved out of caller memory.
// Measured (us a step, operator by operator -> one call): 1 token, H 2048, E
// 128, forward 89 -> 42; training step of 2048 tokens, H 1024, I 2048, E 8
// 817 -> 605.
#include "smoe_layer.h"

using namespace smoe;

namespace {

// Carves 256-byte aligned pieces out of a buffer; with base NULL it only
// counts.
struct Carver {
  uint8_t* base;
  size_t at = 0;
  template <class T>
  void take(T*& p, size_t n) {
    if (base) p = (T*)(base + at);
    at += (n * sizeof(T) + 255) / 256 * 256;
  }
};

struct Dims {
  size_t R, Hp, Ip, Gh, Gi;
  Dims(int T, int H, int I, int K)
      : R((size_t)T * K), Hp(pad128(H)), Ip(pad128(I)), Gh(Hp / kGroup), Gi(Ip / kGroup) {}
};

bool bad_shape(int T, int H, int I, int E, int K) {
  return T <= 0 || H <= 0 || I <= 0 || E <= 0 || K <= 0 || (long long)T * K > 0x7fffffffLL;
}

// fc1 with SwiGLU in its epilogue: the forms that have one
bool fused_swiglu(int I, int flags) {
  if (I % kGroup) return false;
  return !(flags & SMOE_LAYER_POW2) || (flags & SMOE_LAYER_W1_PACKED);
}

void carve_forward(Carver& c, smoe_layer_fwd& a) {
  const Dims d(a.T, a.H, a.I, a.K);
  c.take(a.topk_idx, d.R);
  c.take(a.topk_w, d.R);
  c.take(a.row_map, d.R);
  c.take(a.inv_map, d.R);
  c.take(a.counts, a.E);
  c.take(a.offsets, (size_t)a.E + 1);
  c.take(a.xq, d.R * d.Hp);
  c.take(a.xs, d.R * d.Gh);
  if (!fused_swiglu(a.I, a.flags)) c.take(a.c1, d.R * 2 * a.I);
  c.take(a.hq, d.R * d.Ip);
  c.take(a.hs, d.R * d.Gi);
  c.take(a.y, d.R * a.H);
}

int gemm(const uint8_t* a, const float* as, const uint8_t* w, const float* ws, const int32_t* offsets,
         int E, int R, int N, int Kd, uint16_t* c, bool packed, bool pow2, void* stream) {
  if (!packed) return smoe_grouped_gemm_fp8(a, as, w, ws, offsets, E, R, N, Kd, c, nullptr, 0, stream);
  return pow2 ? smoe_grouped_gemm_fp8_packed_e8m0(a, as, w, ws, offsets, E, R, N, Kd, c, stream)
              : smoe_grouped_gemm_fp8_packed(a, as, w, ws, offsets, E, R, N, Kd, c, stream);
}

#define SMOE_STEP(call)          \
  do {                           \
    const int st__ = (call);     \
    if (st__) return st__;       \
  } while (0)

struct BwdScratch {
  uint8_t *dcq, *dcTq, *hTq, *xTq, *dyTq;
  float *dcs, *dcTs, *hTs, *xTs, *dyTs;
  uint16_t* dc1;
  int32_t* pad;
};

void carve_backward(Carver& m, BwdScratch& b, int T, int H, int I, int E, int K, int ld) {
  const Dims d(T, H, I, K);
  const size_t g = (size_t)ld / kGroup, N = 2 * (size_t)I, Np = pad128(2 * I);
  m.take(b.pad, (size_t)E + 1);
  m.take(b.dcq, d.R * Np);
  m.take(b.dcs, d.R * (Np / kGroup));
  m.take(b.dcTq, N * ld);
  m.take(b.dcTs, N * g);
  if (I % kGroup) m.take(b.dc1, d.R * N);
  m.take(b.hTq, (size_t)I * ld);
  m.take(b.hTs, (size_t)I * g);
  m.take(b.xTq, (size_t)H * ld);
  m.take(b.xTs, (size_t)H * g);
  m.take(b.dyTq, (size_t)H * ld);
  m.take(b.dyTs, (size_t)H * g);
}

// waiter's later work runs after waited's earlier work
int wait_stream(hipStream_t waiter, hipStream_t waited) {
  hipEvent_t ev;
  hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  if (e != hipSuccess) return (int)e;
  e = hipEventRecord(ev, waited);
  if (e == hipSuccess) e = hipStreamWaitEvent(waiter, ev, 0);
  const hipError_t d = hipEventDestroy(ev);  // released once it has completed
  return (int)(e != hipSuccess ? e : d);
}

}  // namespace

extern "C" size_t smoe_layer_forward_scratch_size(int T, int H, int I, int E, int K, int flags) {
  if (bad_shape(T, H, I, E, K)) return 0;
  smoe_layer_fwd a = {};
  a.T = T, a.H = H, a.I = I, a.E = E, a.K = K, a.flags = flags;
  Carver c{nullptr};
  carve_forward(c, a);
  return c.at;
}

extern "C" int smoe_layer_forward(const smoe_layer_fwd* args, void* stream) {
  if (!args) return SMOE_EINVAL_NULL;
  smoe_layer_fwd a = *args;
  if (bad_shape(a.T, a.H, a.I, a.E, a.K)) return SMOE_EINVAL_DIM;
  const bool save = a.scratch == nullptr;
  const bool pow2 = a.flags & SMOE_LAYER_POW2;
  const bool p1 = a.flags & SMOE_LAYER_W1_PACKED, p2 = a.flags & SMOE_LAYER_W2_PACKED;
  if (!save) {
    if ((uintptr_t)a.scratch & 15u) return SMOE_EINVAL_PTRALIGN;
    if (a.scratch_bytes < smoe_layer_forward_scratch_size(a.T, a.H, a.I, a.E, a.K, a.flags))
      return SMOE_EINVAL_WORKSPACE;
    Carver c{(uint8_t*)a.scratch};
    carve_forward(c, a);
  }
  const int R = a.T * a.K, Hp = pad128(a.H), Ip = pad128(a.I);
  const int mode = pow2 ? SMOE_SCALE_POW2 : SMOE_SCALE_AMAX;
  SMOE_STEP(smoe_route_dispatch(a.x, a.logits, a.w_gate, a.bias, a.T, a.H, a.E, a.K, a.topk_idx, a.topk_w,
                                a.row_map, a.inv_map, a.counts, a.offsets, a.xq, a.xs, mode, a.ws,
                                a.ws_bytes, stream));
  if (save || !fused_swiglu(a.I, a.flags)) {
    // the backward needs c1 and bf16 h; without the fused epilogue c1 exists anyway
    SMOE_STEP(gemm(a.xq, a.xs, a.w1, a.w1s, a.offsets, a.E, R, 2 * a.I, Hp, a.c1, p1, pow2, stream));
    SMOE_STEP(smoe_swiglu_quant_ex(a.c1, R, a.I, a.hq, a.hs, save ? a.h : nullptr, mode, stream));
  } else if (pow2) {
    SMOE_STEP(smoe_grouped_gemm_fp8_packed_e8m0_swiglu(a.xq, a.xs, a.w1, a.w1s, a.offsets, a.E, R, a.I, Hp,
                                                       a.hq, a.hs, nullptr, stream));
  } else if (p1) {
    SMOE_STEP(smoe_grouped_gemm_fp8_packed_swiglu(a.xq, a.xs, a.w1, a.w1s, a.offsets, a.E, R, a.I, Hp, a.hq,
                                                  a.hs, nullptr, stream));
  } else {
    SMOE_STEP(smoe_grouped_gemm_fp8_swiglu(a.xq, a.xs, a.w1, a.w1s, a.offsets, a.E, R, a.I, Hp, a.hq, a.hs,
                                           nullptr, stream));
  }
  SMOE_STEP(gemm(a.hq, a.hs, a.w2, a.w2s, a.offsets, a.E, R, a.H, Ip, a.y, p2, pow2, stream));
  return smoe_unpermute_combine(a.y, a.inv_map, a.topk_w, a.T, a.K, a.H, a.out, stream);
}

extern "C" size_t smoe_layer_backward_scratch_size(int T, int H, int I, int E, int K) {
  if (bad_shape(T, H, I, E, K)) return 0;
  const int ld = smoe_quant_cols_ld(T * K, E);
  if (!ld) return 0;
  BwdScratch b;
  Carver m{nullptr};
  carve_backward(m, b, T, H, I, E, K, ld);
  return m.at;
}

extern "C" int smoe_layer_backward(const smoe_layer_bwd* args, void* stream, void* side_stream) {
  if (!args) return SMOE_EINVAL_NULL;
  const smoe_layer_bwd& a = *args;
  if (bad_shape(a.T, a.H, a.I, a.E, a.K)) return SMOE_EINVAL_DIM;
  const int T = a.T, H = a.H, I = a.I, E = a.E, K = a.K, R = T * K;
  const int ld = smoe_quant_cols_ld(R, E);
  if (!ld) return SMOE_EINVAL_DIM;
  if (!a.scratch || !a.offsets) return SMOE_EINVAL_NULL;
  if ((uintptr_t)a.scratch & 15u) return SMOE_EINVAL_PTRALIGN;
  if (E > SMOE_MAX_EXPERTS) return SMOE_EINVAL_EXPERTS;
  if (a.scratch_bytes < smoe_layer_backward_scratch_size(T, H, I, E, K))
    return SMOE_EINVAL_WORKSPACE;
  BwdScratch b = {};
  Carver m{(uint8_t*)a.scratch};
  carve_backward(m, b, T, H, I, E, K, ld);
  const bool pow2 = a.flags & SMOE_LAYER_POW2;
  const bool p1 = a.flags & SMOE_LAYER_W1_PACKED, p2 = a.flags & SMOE_LAYER_W2_PACKED;
  const int cs = a.flags & SMOE_LAYER_COL_POW2 ? SMOE_COLSCALE_POW2 : SMOE_COLSCALE_FP32;
  const int rcs = cs | (pow2 ? SMOE_ROWSCALE_POW2 : 0);
  const int Hp = pad128(H), Np = pad128(2 * I);
  hipStream_t main = (hipStream_t)stream, side = (hipStream_t)side_stream;

  // the padded segment starts of every column quantiser and wgrad
  pad_offsets_launch(a.offsets, E, b.pad, main);
  SMOE_STEP(wait_stream(side, main));
  const int st = [&]() -> int {
    // the wgrad activation operands depend on the forward only (h, and the
    // sorted tokens gathered inside the quantiser); dy's columns are rebuilt
    // from dout, so the fc2 wgrad needs nothing of the caller's stream either
    SMOE_STEP(quant_cols_128x1(a.h, nullptr, 1, R, I, a.offsets, E, ld, b.hTq, b.hTs, b.pad, false, cs, side));
    SMOE_STEP(quant_cols_128x1(a.x, a.row_map, K, R, H, a.offsets, E, ld, b.xTq, b.xTs, b.pad, false, cs, side));
    SMOE_STEP(combine_bwd_quant_cols(a.dout, a.row_map, a.topk_w, T, K, H, a.offsets, E, ld, b.dyTq, b.dyTs,
                                     b.pad, false, cs, side));
    SMOE_STEP(smoe_grouped_gemm_fp8_wgrad_ex(b.dyTq, b.dyTs, b.hTq, b.hTs, b.pad, E, H, I, ld, a.dw2,
                                             a.wgrad2_mode, side));
    // combine backward with dy's 1x128 rows; dy itself is never stored
    SMOE_STEP(combine_bwd_quant(a.dout, a.y, a.inv_map, a.row_map, a.topk_w, T, K, H, a.offsets, E, ld, a.dyq,
                                a.dys, nullptr, nullptr, b.pad, false, a.dtopk_w, rcs, main));
    SMOE_STEP(gemm(a.dyq, a.dys, a.w2t, a.w2ts, a.offsets, E, R, I, Hp, a.dh, p2, pow2, main));
    // SwiGLU backward with both quantisations of dc1 (which is stored only
    // where its row groups straddle the dg | du boundary)
    if (I % kGroup == 0) {
      SMOE_STEP(swiglu_bwd_quant(a.c1, a.dh, R, I, a.offsets, E, ld, b.dcq, b.dcs, b.dcTq, b.dcTs, b.pad, false,
                                 nullptr, rcs, main));
    } else {
      SMOE_STEP(smoe_swiglu_bwd(a.c1, a.dh, R, I, b.dc1, main));
      SMOE_STEP(quant_rows_cols(b.dc1, R, 2 * I, a.offsets, E, ld, b.dcq, b.dcs, b.dcTq, b.dcTs, b.pad, false, rcs,
                                main));
    }
    SMOE_STEP(wait_stream(side, main));
    SMOE_STEP(smoe_grouped_gemm_fp8_wgrad_ex(b.dcTq, b.dcTs, b.xTq, b.xTs, b.pad, E, 2 * I, H, ld, a.dw1,
                                             a.wgrad1_mode, side));
    SMOE_STEP(gemm(b.dcq, b.dcs, a.w1t, a.w1ts, a.offsets, E, R, H, Np, a.dxs, p1, pow2, main));
    SMOE_STEP(combine_launch(a.dxs, a.inv_map, nullptr, T, K, H, a.dx, main));
    // renormalisation + softmax backward into the logits
    return smoe_router_topk_bwd(a.logits, a.topk_idx, a.dtopk_w, T, E, K, a.dlogits, main);
  }();
  // the side stream's work uses the stream's memory: joined also after an error
  const int join = st || !(a.flags & SMOE_LAYER_NO_JOIN) ? wait_stream(main, side) : SMOE_OK;
  return st ? st : join;
}
