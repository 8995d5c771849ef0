// What the f32 projections that multiply pairs of f16 (gemm.h) from LDS share
// (the triangle's and the outer-product mean's): a LayerNorm that leaves rows of
// pairs in LDS, and weights in MFMA fragment order.
#pragma once

#include "gemm.h"

namespace afhip {
namespace {

constexpr int kPairRows = 64;  // rows a workgroup normalises

// Element (n, k) of a weight matrix of `steps` 16-wide steps, in the order the
// lanes load fragments: [n / 32][step][plane][lane][8], lane = n % 32 +
// 32 (k % 16 / 8). h is plane 0; l lies 512 halves on.
__device__ __forceinline__ int64_t pair_fragment(int n, int k, int steps) {
  return (((int64_t)(n >> 5) * steps + (k >> 4)) * 2 * 64 + (n & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
}

// Four lanes normalise one row of cz <= 16 MAXSTEPS channels (a pointer, or null for zeros) and write
// x_hat x_scale as pairs to `dst` (a pair row in LDS): lane `part` takes
// channels 16 i + 4 part + [0, 4) of each block i.
template <typename ZT, int MAXSTEPS>
__device__ __forceinline__ void pair_normalize_row(const ZT* row, int cz, int steps, float eps, float x_scale, int part,
                                                   bool vec, half_t* dst) {
  float v[MAXSTEPS][4];
#pragma unroll
  for (int i = 0; i < MAXSTEPS; i++) {
    const int c = 16 * i + 4 * part;
#pragma unroll
    for (int e = 0; e < 4; e++) v[i][e] = 0.0f;
    if (i >= steps || !row) continue;
    if (vec) {
      if (c < cz) {
        typedef ZT zt4 __attribute__((ext_vector_type(4)));
        const zt4 w = *reinterpret_cast<const zt4*>(row + c);
#pragma unroll
        for (int e = 0; e < 4; e++) v[i][e] = (float)w[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (c + e < cz) v[i][e] = (float)row[c + e];
    }
  }
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < MAXSTEPS; i++) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
  s += __shfl_xor(s, 1);
  s += __shfl_xor(s, 2);
  const float mean = s / (float)cz;
  float d2 = 0.0f;
#pragma unroll
  for (int i = 0; i < MAXSTEPS; i++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v[i][e] = 16 * i + 4 * part + e < cz ? v[i][e] - mean : 0.0f;
      d2 += v[i][e] * v[i][e];
    }
  d2 += __shfl_xor(d2, 1);
  d2 += __shfl_xor(d2, 2);
  const float rstd = fast_rsqrt(d2 / (float)cz + eps) * x_scale;
#pragma unroll
  for (int i = 0; i < MAXSTEPS; i++) {
    if (i >= steps) continue;
    half2v h0, l0, h1, l1;
    pair_split2(v[i][0] * rstd, v[i][1] * rstd, h0, l0);
    pair_split2(v[i][2] * rstd, v[i][3] * rstd, h1, l1);
    half_t* p = dst + 32 * i + 4 * part;
    *reinterpret_cast<half4*>(p) = half4{h0[0], h0[1], h1[0], h1[1]};
    *reinterpret_cast<half4*>(p + 16) = half4{l0[0], l0[1], l1[0], l1[1]};
  }
}

// Two steps' fragments (h, l of each) of one matrix block; `w` at the block's
// first fragment, this lane's 16 bytes.
struct PairFragments {
  half8 h[2], l[2];
  __device__ __forceinline__ void load(const half_t* w, int s) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      h[u] = *reinterpret_cast<const half8*>(w + (int64_t)(s + u) * 1024);
      l[u] = *reinterpret_cast<const half8*>(w + (int64_t)(s + u) * 1024 + 512);
    }
  }
};

// LDS pair rows of 16 `steps` channels, padded by 16 bytes: 16 rows' fragments
// then start on 16 different groups of four banks.
__host__ __device__ constexpr int pair_pitch(int steps) { return 32 * steps + 8; }  // halves

// Rows whose four-channel chunks load at once.
inline bool rows_on_four(const void* x, int channels, size_t es) {
  return channels % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & (4 * es - 1)) == 0;
}

}  // namespace
}  // namespace afhip
