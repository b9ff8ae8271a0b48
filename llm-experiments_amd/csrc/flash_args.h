// Arguments of the fp32 flash kernels (flash_fp32.hip, flash_split.hip).
#pragma once

#include "skv_common.h"

namespace skv {

struct FfwdArgs {
  const float* q;  // [B, C, Hq, D]
  const float* k;  // [B, T_cap, Hkv, D]
  const float* v;
  const int32_t* start;  // per-sequence position of query 0 (NULL: 0)
  const int32_t* n_new;  // per-sequence valid queries (NULL: C)
  float* out;            // [B, C, Hq, D]; rows i >= n_new[b] get zeros
  float* L;              // [B, C, Hq] softmax sums (may be NULL)
  float* M;              // [B, C, Hq] row maxima of the scaled scores (may be NULL)
  int C, Hq, Hkv, T_cap, BH, n_blocks;
  int D;  // head dim (the padded size is the kernel's template D)
  float sl2;  // scale * log2(e)
};

struct FbwdArgs {
  const float* q;
  const float* k;
  const float* v;
  const float* o;
  const float* dout;
  const float* L;
  const float* M;
  float* dq;
  float* dk;
  float* dv;
  float* delta;  // [B, N, H] row deltas Dl
  float* ds;     // dS in 32 x 32 tiles (five-product form), or NULL
  int N, H, BH, n_blocks;
  int D;  // head dim (the padded size is the kernel's template D)
  float scale, sl2;  // scale and scale * log2(e)
};

// Padded head dim and load mode of a head dim: a multiple of 16 up to 128,
// then 192 or 256. Mode 0: the padded size is the head dim (16-byte vectors
// throughout); 1: D % 4 == 0 (float4 loads, groups past D read as zeros); 2:
// any other D (element loads).
struct FlashShape {
  int DP, mode;
};
inline FlashShape flash_shape(int D) {
  const int DP = D <= 128 ? (D + 15) / 16 * 16 : D <= 192 ? 192 : 256;
  return {DP, D == DP ? 0 : (D % 4 == 0 ? 1 : 2)};
}

// Expands X(DP, MODE) for every kernel shape up to 128.
#define SKV_FLASH_SHAPES(X)                                                           \
  X(16, 0) X(16, 1) X(16, 2) X(32, 0) X(32, 1) X(32, 2) X(48, 0) X(48, 1) X(48, 2)    \
  X(64, 0) X(64, 1) X(64, 2) X(80, 0) X(80, 1) X(80, 2) X(96, 0) X(96, 1) X(96, 2)    \
  X(112, 0) X(112, 1) X(112, 2) X(128, 0) X(128, 1) X(128, 2)

// Four consecutive elements c..c+3 of a row with D elements, zeros past D.
typedef float flash_f32x4 __attribute__((ext_vector_type(4)));
template <int MODE>
__device__ __forceinline__ flash_f32x4 load4m(const float* row, int c, int D) {
  if constexpr (MODE == 0) {
    return *reinterpret_cast<const flash_f32x4*>(row + c);
  } else if constexpr (MODE == 1) {
    const bool ok = c < D;  // D % 4 == 0: the group lies wholly inside or past D
    const flash_f32x4 x = *reinterpret_cast<const flash_f32x4*>(row + (ok ? c : 0));
    return ok ? x : flash_f32x4{0.f, 0.f, 0.f, 0.f};
  } else {
    flash_f32x4 x;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bool ok = c + t < D;
      const float v = row[ok ? c + t : 0];
      x[t] = ok ? v : 0.f;
    }
    return x;
  }
}

// Stores the elements c..c+3 of y that lie inside a row of D elements.
template <int MODE>
__device__ __forceinline__ void store4m(float* row, int c, int D, const flash_f32x4& y) {
  if constexpr (MODE == 2) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (c + t < D) row[c + t] = y[t];
  } else {
    if (c < D) *reinterpret_cast<flash_f32x4*>(row + c) = y;
  }
}

// The forward up to a padded head dim of 128 (flash_split.hip).
int flash_fwd_split(const FfwdArgs& a, hipStream_t s, const char* fn);
// The backward: five products where a.ds is set (head dims up to 64, a.delta
// already written), else seven.
int flash_bwd_split(const FbwdArgs& a, hipStream_t s, const char* fn);

}  // namespace skv
