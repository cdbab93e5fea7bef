// smoe_layer.h — launches the layer entry points (smoe_layer.hip) share with
// the single-operator entry points, in forms only the layer uses: the padded
// segment starts computed once for all quantisers, and a combine without
// weights.  Each checks its arguments as its entry point does.
#pragma once

#include "smoe_common.h"

namespace smoe {

// out[t] = the sum of token t's rows of y, weighted by w unless w is NULL.
int combine_launch(const uint16_t* y, const int32_t* inv_map, const float* w, int T, int K, int H,
                   uint16_t* out, void* stream);

// make_pad: fill pad from offsets first; otherwise pad already holds it.
int quant_cols_128x1(const uint16_t* x, const int32_t* gather, int gather_div, int R, int C,
                     const int32_t* offsets, int E, int ld, uint8_t* xTq, float* xTs, int32_t* pad,
                     bool make_pad, int col_scale, void* stream);
int quant_rows_cols(const uint16_t* x, int R, int C, const int32_t* offsets, int E, int ld,
                    uint8_t* xq, float* xs, uint8_t* xTq, float* xTs, int32_t* pad, bool make_pad,
                    int col_scale, void* stream);
int swiglu_bwd_quant(const uint16_t* c1, const uint16_t* dh, int R, int I, const int32_t* offsets,
                     int E, int ld, uint8_t* dcq, float* dcs, uint8_t* dcTq, float* dcTs,
                     int32_t* pad, bool make_pad, uint16_t* dc1, int col_scale, void* stream);
int combine_bwd_quant(const uint16_t* dout, const uint16_t* y, const int32_t* inv_map,
                      const int32_t* row_map, const float* w, int T, int K, int H,
                      const int32_t* offsets, int E, int ld, uint8_t* dyq, float* dys,
                      uint8_t* dyTq, float* dyTs, int32_t* pad, bool make_pad, float* dw,
                      int col_scale, void* stream);
int combine_bwd_quant_cols(const uint16_t* dout, const int32_t* row_map, const float* w, int T,
                           int K, int H, const int32_t* offsets, int E, int ld, uint8_t* dyTq,
                           float* dyTs, int32_t* pad, bool make_pad, int col_scale, void* stream);
void pad_offsets_launch(const int32_t* offsets, int E, int32_t* pad, hipStream_t s);

}  // namespace smoe
