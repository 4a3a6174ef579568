// What nv_linear is called with, and its element-wise functions: shared by linear.hip and linear_deep.hip.
#pragma once
#include "anyt.h"

struct LinArgs {
  const void* a;
  int64_t a_rs;
  const int32_t* a_rows;
  const void* w;
  int64_t w_rs;
  const void* bias;
  void* out;
  int64_t out_rs;
  int64_t M;
  int N, K;
  int64_t a_bs, w_bs, out_bs, bias_bs;
  const int32_t* group_off;
  const float* epi_ptr;
  int64_t epi_rs;
  float epi_c;
  int act;
  int vec_a, vec_w;
  const float* row_scale;    // [output rows] factor of the product, ahead of bias and epilogue, or null
};

enum { EPI_NONE = 0, EPI_GLU = 1, EPI_SOFTCAP = 2, EPI_ROW_GATE = 3, EPI_ACT = 4 };

// EPI_ACT: an element-wise function of the product.  act 0 SiLU, 1 tanh-form GELU, 2 xIELU with its two positive
// coefficients at epi_ptr (a z^2 + z/2 above zero, b (exp(z) - 1 - z) + z/2 below), 3 multiplication by epi_c, 4 erf-form
// GELU.
__device__ __forceinline__ float unary_act(float v, int act, const float* prm, float c) {
  switch (act) {
    case 0: return silu_f32(v);
    case 1: return gelu_tanh_f32(v);
    case 2: return v > 0.0f ? prm[0] * v * v + 0.5f * v : prm[1] * (expm1f(v) - v) + 0.5f * v;
    case 4: return gelu_erf_f32(v);
    default: return v * c;
  }
}

// 16-bit products on the tiles of stream_deep.h (linear_deep.hip); total_rows: of all groups
hipError_t linear_deep_launch(const LinArgs& p, int epilogue, bool out_16bit, int64_t total_rows, int batch, hipStream_t s);
// the same on those of stream_tiles.h (linear_eight.hip)
hipError_t linear_eight_launch(const LinArgs& p, int epilogue, bool out_16bit, int64_t total_rows, int batch, hipStream_t s);
// fp32 products as sums of 16-bit ones (linear_split.hip), in tiles of 64, 128 or 256 rows by 128 columns
enum { SPLIT_64 = 0, SPLIT_128 = 1, SPLIT_256 = 2 };
hipError_t linear_split_launch(const LinArgs& p, int epilogue, bool out_16bit, int64_t total_rows, int batch, int tile, hipStream_t s);
