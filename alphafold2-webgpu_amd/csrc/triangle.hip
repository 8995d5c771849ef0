// Triangle multiplication (outgoing and incoming) for gfx950.
//
// Three launches per output block, replacing the reference's seven kernels
// (src/triangle/shaders.ts:151-589):
//
//  1. tri_project: LayerNorm of 64 pair rows in LDS, the four projections
//     (a, a-gate, b, b-gate) on MFMA, the gated product a = mask*(x+b)*sig(g+bg)
//     staged through LDS and stored channel-major as [c][row]. The direction
//     is folded into which pair a row reads: outgoing row r is pair r;
//     incoming row r = j*L + k reads pair (k, j). Both directions therefore
//     leave the contraction the same NT problem.
//  2. the contraction: one batched GEMM over the hidden channels through the
//     shared tiled GEMM, out[c][i][j] = sum_k R[c][i][k] C[c][j][k] with
//     (R, C) = (a, b) outgoing, (b, a) incoming. That is AlphaFold's
//     "ikc,jkc->ijc" and "kjc,kic->ijc" (src/triangle/shaders.ts:452-495).
//  3. tri_output: the contracted tile (channel-major, 64 pairs) is normalised
//     over the hidden channels in LDS and projected by linearZ; the same pairs
//     of z are normalised and projected by linearG; out = (p + bz)*sig(g + bg).
//     The gate is recomputed here from z rather than stored and re-read.
//
// At f32 precision with 64 channels or more 1 and 3 multiply pairs of f16 on the
// f16 MFMA (gemm.h; the tri_*_pair kernels below); the contraction is the f32 GEMM.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "gemm.h"
#include "pairs.h"
#include "triangle_fast.h"

namespace afhip {

namespace {

constexpr int kRows = 64;  // pair rows per workgroup in the projection kernels
constexpr int kC = 128;    // the fast path's c_z = c_hidden

// The projections' products. f32 precision multiplies pairs of f16 where both
// of its sums are long enough (gemm.h).
enum class Products { kF16, kF32, kPairs };
bool tri_pairs(const afhip_triangle_desc& d) {
  return d.precision == AFHIP_PRECISION_F32 && std::min(d.c_z, d.c_hidden) >= kPairMinK;
}

struct TriWeights {
  // Offsets in bytes into the prepared buffer.
  size_t ln_in_w, ln_in_b, w_proj, b_proj, ln_out_w, ln_out_b, w_z, b_z, w_g, b_g;
  size_t fold_w, fold_b;  // the f16 fast path's folded weights (0 when not eligible)
  size_t s_proj, s_z, s_g;  // over pairs: output scales of the pair products
  size_t total;
  int czp, chp, czo;  // padded input width (multiple of 32), padded hidden, padded output rows
};

TriWeights tri_layout(const afhip_triangle_desc& d) {
  TriWeights w{};
  size_t es = d.precision == AFHIP_PRECISION_F16 ? 2 : 4;
  w.czp = (int)round_up(d.c_z, 32);
  w.chp = (int)round_up(d.c_hidden, 32);
  w.czo = (int)round_up(d.c_z, 32);
  size_t at = 0;
  auto take = [&](size_t bytes) {
    size_t here = at;
    at = round_up((int64_t)(at + bytes), 256);
    return here;
  };
  if (!tri_pairs(d)) {  // the pair products' weights hold the LayerNorms' affines
    w.ln_in_w = take(4 * (size_t)d.c_z);
    w.ln_in_b = take(4 * (size_t)d.c_z);
    w.ln_out_w = take(4 * (size_t)d.c_hidden);
    w.ln_out_b = take(4 * (size_t)d.c_hidden);
  }
  w.w_proj = take(es * 4 * (size_t)w.chp * w.czp);
  w.b_proj = take(4 * 4 * (size_t)w.chp);
  w.w_z = take(es * (size_t)w.czo * w.chp);
  w.b_z = take(4 * (size_t)w.czo);
  w.w_g = take(es * (size_t)w.czo * w.czp);
  w.b_g = take(4 * (size_t)w.czo);
  if (tri_pairs(d)) {
    w.s_proj = take(4 * 4 * (size_t)w.chp);
    w.s_z = take(4 * (size_t)w.czo);
    w.s_g = take(4 * (size_t)w.czo);
  }
  if (triangle_fast_eligible(d)) {
    w.fold_w = take(2 * (size_t)kFoldMatrices * d.c_z * d.c_z);
    w.fold_b = take(4 * (size_t)kFoldMatrices * d.c_z);
  }
  w.total = at;
  return w;
}

struct TriWorkspace {
  size_t op_a, op_b, contracted, total;
  int64_t cstride;  // elements between channels of an operand
  int64_t bstride;  // elements between channels of the contracted block
  int block_rows;
};

TriWorkspace tri_workspace(const afhip_triangle_desc& d) {
  TriWorkspace w{};
  size_t es = d.precision == AFHIP_PRECISION_F16 ? 2 : 4;
  int64_t L = d.length, P = L * L;
  w.block_rows = d.block_rows > 0 ? std::min(d.block_rows, d.length) : d.length;
  // The fast output kernels address a block's z, contracted values and
  // output with 32-bit buffer offsets: at long lengths the block shrinks to
  // what they reach (the result does not depend on the block).
  if (triangle_fast_eligible(d)) w.block_rows = std::min(w.block_rows, triangle_fast_block_rows(d));
  w.cstride = round_up(P, 64);
  w.bstride = round_up((int64_t)w.block_rows * L, 64);
  size_t at = 0;
  auto take = [&](size_t bytes) {
    size_t here = at;
    at = round_up((int64_t)(at + bytes), 256);
    return here;
  };
  w.op_a = take(es * (size_t)d.c_hidden * w.cstride);
  w.op_b = take(es * (size_t)d.c_hidden * w.cstride);
  w.contracted = take(es * (size_t)d.c_hidden * w.bstride);
  w.total = at;
  return w;
}

// ---------------------------------------------------------------------------
// Shared LDS helpers
// ---------------------------------------------------------------------------

// Mean and 1/sigma over `channels` of 64 columns of a channel-major f32 tile
// (xs[c * pitch + q]); four lanes per column, two-pass as the reference's
// statistics kernels compute them (shaders.ts:242-281, :501-522).
__device__ __forceinline__ void column_stats(const float* xs, int pitch, int channels, float eps, int tid,
                                             float& mean, float& rstd) {
  const int q = tid >> 2, part = tid & 3;
  float s = 0.0f;
  for (int c = part; c < channels; c += 4) s += xs[c * pitch + q];
  s += __shfl_xor(s, 1);
  s += __shfl_xor(s, 2);
  mean = s / (float)channels;
  float v = 0.0f;
  for (int c = part; c < channels; c += 4) {
    float d = xs[c * pitch + q] - mean;
    v += d * d;
  }
  v += __shfl_xor(v, 1);
  v += __shfl_xor(v, 2);
  rstd = fast_rsqrt(v / (float)channels + eps);
}

template <typename T> __device__ __forceinline__ float ldf(const T* p) { return (float)*p; }

// ---------------------------------------------------------------------------
// 1. Gated projections
// ---------------------------------------------------------------------------

struct ProjectArgs {
  const void* z;
  const float* mask;
  const float* ln_w;
  const float* ln_b;
  const void* w_proj;  // [4][chp][czp]: ap, ag, bp, bg (the pair kernels': in fragment order)
  const float* b_proj; // [4][chp]
  const float* s_proj; // [4][chp] (pair kernels)
  void* out_a;
  void* out_b;
  int64_t cstride;
  int L, P, cz, ch, czp, chp;
  int incoming;
  float eps;
  float x_scale;  // the pair kernels hold x_hat times this
};

template <typename ZT, bool F16MATH>
__global__ __launch_bounds__(256) void tri_project_kernel(ProjectArgs a) {
  using CT = typename std::conditional<F16MATH, half_t, float>::type;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // xs: f32 [czp][kRows + 1], channel-major raw z; an: CT [kRows][czp + 8] (f16 only);
  // stage: CT [64][kRows + 8] output transpose.
  const int xpitch = kRows + 1;
  float* xs = reinterpret_cast<float*>(smem);
  size_t off = round_up((int64_t)a.czp * xpitch * 4, 16);
  CT* an = reinterpret_cast<CT*>(smem + off);
  const int apitch = a.czp + 8;
  if (F16MATH) off += round_up((int64_t)kRows * apitch * 2, 16);
  CT* stage = reinterpret_cast<CT*>(smem + off);
  constexpr int spitch = kRows + 8;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = blockIdx.x * kRows;
  const ZT* z = reinterpret_cast<const ZT*>(a.z);

  // Load 64 pair rows, transposed to channel-major in LDS.
  for (int idx = tid; idx < kRows * a.czp; idx += 256) {
    const int i = idx / a.czp, c = idx - i * a.czp;
    const int r = r0 + i;
    float v = 0.0f;
    if (r < a.P && c < a.cz) {
      const int p = a.incoming ? (r % a.L) * a.L + r / a.L : r;
      v = ldf(z + (int64_t)p * a.cz + c);
    }
    xs[c * xpitch + i] = v;
  }
  __syncthreads();
  float mean, rstd;
  column_stats(xs, xpitch, a.cz, a.eps, tid, mean, rstd);
  {
    const int q = tid >> 2, part = tid & 3;
    for (int c = part; c < a.czp; c += 4) {
      float v = c < a.cz ? (xs[c * xpitch + q] - mean) * rstd * a.ln_w[c] + a.ln_b[c] : 0.0f;
      if (F16MATH) an[q * apitch + c] = (CT)v;
      else xs[c * xpitch + q] = v;
    }
  }
  __syncthreads();

  const CT* W = reinterpret_cast<const CT*>(a.w_proj);
  const int rw = 32 * (wave & 1);
  for (int o = 0; o < 2; o++) {
    const CT* wp = W + (size_t)(2 * o) * a.chp * a.czp;
    const CT* wg = W + (size_t)(2 * o + 1) * a.chp * a.czp;
    const float* bp = a.b_proj + (2 * o) * a.chp;
    const float* bg = a.b_proj + (2 * o + 1) * a.chp;
    CT* out = reinterpret_cast<CT*>(o == 0 ? a.out_a : a.out_b);
    for (int h0 = 0; h0 < a.chp; h0 += 64) {
      const int hc = h0 + 32 * (wave >> 1);
      if (hc < a.chp) {
        floatx16 accp, accg;
#pragma unroll
        for (int v = 0; v < 16; v++) accp[v] = accg[v] = 0.0f;
        const int n = hc + (lane & 31);
        if constexpr (F16MATH) {
          for (int k = 0; k < a.czp; k += 16) {
            const int kk = k + 8 * (lane >> 5);
            half8 af = *reinterpret_cast<const half8*>(an + (rw + (lane & 31)) * apitch + kk);
            half8 bpf = *reinterpret_cast<const half8*>(wp + (size_t)n * a.czp + kk);
            half8 bgf = *reinterpret_cast<const half8*>(wg + (size_t)n * a.czp + kk);
            accp = mfma_f16(af, bpf, accp);
            accg = mfma_f16(af, bgf, accg);
          }
        } else {
          for (int k = 0; k < a.czp; k += 2) {
            const int kk = k + (lane >> 5);
            float af = xs[kk * xpitch + rw + (lane & 31)];
            accp = mfma_f32(af, wp[(size_t)n * a.czp + kk], accp);
            accg = mfma_f32(af, wg[(size_t)n * a.czp + kk], accg);
          }
        }
        const float bpv = bp[n], bgv = bg[n];
#pragma unroll
        for (int v = 0; v < 16; v++) {
          const int i = rw + mfma_row(v, lane);
          const int r = r0 + i;
          float val = 0.0f;
          if (r < a.P) {
            const int p = a.incoming ? (r % a.L) * a.L + r / a.L : r;
            val = a.mask[p] * (accp[v] + bpv) * sigmoidf_(accg[v] + bgv);
          }
          stage[(n - h0) * spitch + i] = (CT)val;
        }
      }
      __syncthreads();
      // 64 channels x 64 rows, written along the rows of each channel.
      for (int idx = tid; idx < 64 * kRows; idx += 256) {
        const int hl = idx / kRows, i = idx - hl * kRows;
        const int h = h0 + hl, r = r0 + i;
        if (h < a.ch && r < a.P) out[(int64_t)h * a.cstride + r] = stage[hl * spitch + i];
      }
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
// 3. Hidden LayerNorm, output projection and gate
// ---------------------------------------------------------------------------

struct OutputArgs {
  const void* contracted;  // CT [ch][bstride], pairs of this block
  int64_t bstride;
  const void* z;
  const float* ln_in_w;
  const float* ln_in_b;
  const float* ln_out_w;
  const float* ln_out_b;
  const void* w_z;  // [czo][chp]
  const float* b_z;
  const void* w_g;  // [czo][czp]
  const float* b_g;
  const float* s_z;  // pair kernels
  const float* s_g;
  void* out;
  int pair0;        // first pair of this block
  int pairs;        // pairs in this block
  int cz, ch, czp, chp;
  int residual;
  int in_place;  // out overlaps z (read by the launch)
  float eps;
  float x_scale, h_scale;  // the pair kernels' x_hat of z and of the contracted values
};

// Loads 64 columns of a channel-major tile (xs[c][q]) and normalises them in
// place (f32) or into an[q][c] (f16). Returns after a barrier.
template <typename CT, bool F16MATH>
__device__ __forceinline__ void normalize_tile(float* xs, int xpitch, CT* an, int apitch, int channels, int padded,
                                               const float* w, const float* b, float eps, int tid) {
  float mean, rstd;
  column_stats(xs, xpitch, channels, eps, tid, mean, rstd);
  const int q = tid >> 2, part = tid & 3;
  __syncthreads();
  for (int c = part; c < padded; c += 4) {
    float v = c < channels ? (xs[c * xpitch + q] - mean) * rstd * w[c] + b[c] : 0.0f;
    if (F16MATH) an[q * apitch + c] = (CT)v;
    else xs[c * xpitch + q] = v;
  }
  __syncthreads();
}

// acc[t] += A (64 x K from LDS) * W^T for the wave's column tiles.
template <typename CT, bool F16MATH>
__device__ __forceinline__ void tile_gemm(floatx16 (&acc)[2], const float* xs, int xpitch, const CT* an, int apitch,
                                          const CT* W, int K, int czo, int lane, int wave) {
  const int rw = 32 * (wave & 1);
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int j = (wave >> 1) + 2 * t;
    if (32 * j >= czo) continue;
    const int n = 32 * j + (lane & 31);
    if constexpr (F16MATH) {
      for (int k = 0; k < K; k += 16) {
        const int kk = k + 8 * (lane >> 5);
        half8 af = *reinterpret_cast<const half8*>(an + (rw + (lane & 31)) * apitch + kk);
        half8 bf = *reinterpret_cast<const half8*>(W + (size_t)n * K + kk);
        acc[t] = mfma_f16(af, bf, acc[t]);
      }
    } else {
      for (int k = 0; k < K; k += 2) {
        const int kk = k + (lane >> 5);
        acc[t] = mfma_f32(xs[kk * xpitch + rw + (lane & 31)], W[(size_t)n * K + kk], acc[t]);
      }
    }
  }
}

template <typename ZT, typename OT, bool F16MATH>
__global__ __launch_bounds__(256) void tri_output_kernel(OutputArgs a) {
  using CT = typename std::conditional<F16MATH, half_t, float>::type;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int xpitch = kRows + 1;
  const int kmax = a.chp > a.czp ? a.chp : a.czp;
  float* xs = reinterpret_cast<float*>(smem);
  CT* an = reinterpret_cast<CT*>(smem + round_up((int64_t)kmax * xpitch * 4, 16));
  const int apitch = kmax + 8;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q0 = blockIdx.x * kRows;
  const CT* X = reinterpret_cast<const CT*>(a.contracted);
  const ZT* z = reinterpret_cast<const ZT*>(a.z);

  // Phase 1: contracted tile, channel-major as stored.
  for (int idx = tid; idx < a.chp * kRows; idx += 256) {
    const int c = idx / kRows, q = idx - c * kRows;
    float v = 0.0f;
    if (c < a.ch && q0 + q < a.pairs) v = (float)X[(int64_t)c * a.bstride + q0 + q];
    xs[c * xpitch + q] = v;
  }
  __syncthreads();
  normalize_tile<CT, F16MATH>(xs, xpitch, an, apitch, a.ch, a.chp, a.ln_out_w, a.ln_out_b, a.eps, tid);
  floatx16 accz[2], accg[2];
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int v = 0; v < 16; v++) accz[t][v] = accg[t][v] = 0.0f;
  tile_gemm<CT, F16MATH>(accz, xs, xpitch, an, apitch, reinterpret_cast<const CT*>(a.w_z), a.chp,
                         (int)round_up(a.cz, 32), lane, wave);
  __syncthreads();

  // Phase 2: the same pairs of z, transposed to channel-major.
  for (int idx = tid; idx < kRows * a.czp; idx += 256) {
    const int q = idx / a.czp, c = idx - q * a.czp;
    float v = 0.0f;
    if (c < a.cz && q0 + q < a.pairs) v = (float)z[(int64_t)(a.pair0 + q0 + q) * a.cz + c];
    xs[c * xpitch + q] = v;
  }
  __syncthreads();
  normalize_tile<CT, F16MATH>(xs, xpitch, an, apitch, a.cz, a.czp, a.ln_in_w, a.ln_in_b, a.eps, tid);
  tile_gemm<CT, F16MATH>(accg, xs, xpitch, an, apitch, reinterpret_cast<const CT*>(a.w_g), a.czp,
                         (int)round_up(a.cz, 32), lane, wave);

  OT* out = reinterpret_cast<OT*>(a.out);
  const int rw = 32 * (wave & 1);
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int j = (wave >> 1) + 2 * t;
    const int n = 32 * j + (lane & 31);
    if (n >= a.cz) continue;
    const float bz = a.b_z[n], bg = a.b_g[n];
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int q = q0 + rw + mfma_row(v, lane);
      if (q >= a.pairs) continue;
      float y = (accz[t][v] + bz) * sigmoidf_(accg[t][v] + bg);
      const int64_t at = (int64_t)(a.pair0 + q) * a.cz + n;
      if (a.residual) y += (float)out[at];
      out[at] = (OT)y;
    }
  }
}

// ---------------------------------------------------------------------------
// f32 precision, c_z and c_hidden >= 64: both projections over pairs of f16
// ---------------------------------------------------------------------------
//
// The f32 kernels above run the f32 MFMA, one 64-pair tile a workgroup
// through all four (two) matrices, with the weights read element by element in
// the middle of the MFMA chain: at L = 59, 55 of 256 CUs worked through 32k
// cycles of MFMA each. Here a tile's columns are split over as many workgroups
// as it takes to fill the chip (every one normalises the tile for itself), the
// products are three f16 MFMAs of 32 cycles where eight f32 ones took 512, and
// the weights come in fragment order, 1 KiB a load, one group of steps ahead.
// Measured at c_z = c_h = 128, project / output: L = 59 83 / 63 us before,
// 10.7 / 12.2 after; L = 256 365 / 157 before, 58 / 64 after.

constexpr int kMaxSteps = 8;  // c_z <= 128 in steps of 16

struct PairSources {
  struct Matrix {
    const float *w, *b, *gamma, *beta;  // w [rows][cols], the LayerNorm that feeds it
    int rows, cols, padded, steps, x_exp;
    half_t* out;
    float *scale, *bias;
  } m[6];
};

// One workgroup a (row, matrix): W' = W diag(gamma) in double times 2^e (the
// largest element in [2^14, 2^15)), scale 2^-(x_exp + e), bias b + W beta;
// padding rows and columns are zeros.
__global__ __launch_bounds__(64) void tri_pair_prepare_kernel(PairSources src) {
  const PairSources::Matrix& m = src.m[blockIdx.y];
  const int n = blockIdx.x, lane = threadIdx.x;
  if (n >= m.padded) return;
  const bool in = n < m.rows;
  const float* w = m.w + (int64_t)n * m.cols;
  float most = 0.0f;
  double offset = 0.0;
  if (in)
    for (int c = lane; c < m.cols; c += 64) {
      most = fmaxf(most, fabsf((float)((double)w[c] * m.gamma[c])));
      offset += (double)w[c] * m.beta[c];
    }
  for (int o = 32; o > 0; o >>= 1) {
    most = fmaxf(most, __shfl_xor(most, o));
    offset += __shfl_xor(offset, o);
  }
  const int e = pair_exponent(most);
  for (int c = lane; c < 16 * m.steps; c += 64) {
    half_t h, l;
    pair_split(in && c < m.cols ? (float)ldexp((double)w[c] * m.gamma[c], e) : 0.0f, h, l);
    const int64_t at = pair_fragment(n, c, m.steps);
    m.out[at] = h;
    m.out[at + 512] = l;
  }
  if (lane == 0) {
    m.scale[n] = in ? ldexpf(1.0f, -(m.x_exp + e)) : 1.0f;
    m.bias[n] = in ? (float)(m.b[n] + offset) : 0.0f;
  }
}

// Wave (rows 32 (w % 2).., operand w / 2) of a tile computes W x_hat^T for the
// projection and the gate of 32 hidden channels: a lane ends with one pair and
// 16 channels, so each store of a channel is 32 consecutive pairs.
template <typename ZT> __global__ __launch_bounds__(256) void tri_project_pair_kernel(ProjectArgs a, int vec) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  half_t* an = reinterpret_cast<half_t*>(smem);
  const int steps = a.czp / 16, pitch = pair_pitch(steps);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = blockIdx.x * kPairRows;
  const ZT* z = reinterpret_cast<const ZT*>(a.z);
  auto pair_of = [&](int r) { return a.incoming ? (r % a.L) * a.L + r / a.L : r; };
  const int o = wave >> 1, hi = lane >> 5;
  const int r = r0 + 32 * (wave & 1) + (lane & 31);
  const float keep = r < a.P ? a.mask[pair_of(r)] : 0.0f;
  const int blocks = a.chp / 32;
  const half_t* W = reinterpret_cast<const half_t*>(a.w_proj) + (int64_t)2 * o * a.chp * 2 * a.czp + 8 * lane;
  const int64_t matrix = (int64_t)a.chp * 2 * a.czp, block = (int64_t)steps * 1024;
  PairFragments fp, fg;
  fp.load(W + blockIdx.y * block, 0);
  fg.load(W + matrix + blockIdx.y * block, 0);
  {
    const int q = tid >> 2, rq = r0 + q;
    pair_normalize_row<ZT, kMaxSteps>(rq < a.P ? z + (int64_t)pair_of(rq) * a.cz : nullptr, a.cz, steps, a.eps, a.x_scale, tid & 3,
                           vec, an + q * pitch);
  }
  __syncthreads();
  const half_t* xr = an + (32 * (wave & 1) + (lane & 31)) * pitch + 8 * hi;
  for (int nb = blockIdx.y; nb < blocks; nb += gridDim.y) {
    floatx16 p = {}, g = {};
    for (int s = 0; s < steps; s += 2) {
      const PairFragments cp = fp, cg = fg;
      // The next two steps, or the next block's first.
      const int ns = s + 2 < steps ? s + 2 : 0, nn = min(s + 2 < steps ? nb : nb + (int)gridDim.y, blocks - 1);
      fp.load(W + nn * block, ns);
      fg.load(W + matrix + nn * block, ns);
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const half8 xh = *reinterpret_cast<const half8*>(xr + 32 * (s + u));
        const half8 xl = *reinterpret_cast<const half8*>(xr + 32 * (s + u) + 16);
        p = mfma_f16(cp.h[u], xh, p);
        g = mfma_f16(cg.h[u], xh, g);
        p = mfma_f16(cp.h[u], xl, p);
        g = mfma_f16(cg.h[u], xl, g);
        p = mfma_f16(cp.l[u], xh, p);
        g = mfma_f16(cg.l[u], xh, g);
      }
    }
    const int c0 = 32 * nb + 4 * hi;
    const float *sp = a.s_proj + 2 * o * a.chp, *bp = a.b_proj + 2 * o * a.chp;
    float* out = reinterpret_cast<float*>(o == 0 ? a.out_a : a.out_b) + r;
#pragma unroll
    for (int v4 = 0; v4 < 4; v4++) {
      const int c = c0 + 8 * v4;
      const float4 s1 = *reinterpret_cast<const float4*>(sp + c), b1 = *reinterpret_cast<const float4*>(bp + c);
      const float4 s2 = *reinterpret_cast<const float4*>(sp + a.chp + c), b2 = *reinterpret_cast<const float4*>(bp + a.chp + c);
      const float S1[4] = {s1.x, s1.y, s1.z, s1.w}, B1[4] = {b1.x, b1.y, b1.z, b1.w};
      const float S2[4] = {s2.x, s2.y, s2.z, s2.w}, B2[4] = {b2.x, b2.y, b2.z, b2.w};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float y = keep * fmaf(p[4 * v4 + e], S1[e], B1[e]) * sigmoidf_(fmaf(g[4 * v4 + e], S2[e], B2[e]));
        if (c + e < a.ch && r < a.P) out[(int64_t)(c + e) * a.cstride] = y;
      }
    }
  }
}

// A tile of 64 pairs of the output: waves 0 and 1 (rows 32 w..) multiply the
// normalised contraction by linearZ, waves 2 and 3 the normalised z by linearG;
// the gates cross through LDS. A lane ends with one channel and 16 pairs, so
// each store of a pair is 32 consecutive channels.
template <typename ZT, typename OT> __global__ __launch_bounds__(256) void tri_output_pair_kernel(OutputArgs a, int vec) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int zsteps = a.czp / 16, hsteps = a.chp / 16, zpitch = pair_pitch(zsteps), hpitch = pair_pitch(hsteps);
  half_t* hn = reinterpret_cast<half_t*>(smem);
  half_t* zn = hn + kPairRows * hpitch;
  float* red = reinterpret_cast<float*>(zn + kPairRows * zpitch);  // [2][4][64], then the gates [2][32][32]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q0 = blockIdx.x * kPairRows;
  const ZT* z = reinterpret_cast<const ZT*>(a.z);
  const float* X = reinterpret_cast<const float*>(a.contracted);
  const bool gate = wave >= 2;
  const int rw = 32 * (wave & 1), blocks = (a.cz + 31) / 32;
  const int steps = gate ? zsteps : hsteps;
  const half_t* W = reinterpret_cast<const half_t*>(gate ? a.w_g : a.w_z) + 8 * lane;
  const int64_t block = (int64_t)steps * 1024;
  PairFragments f;
  f.load(W + blockIdx.y * block, 0);

  // The contraction's LayerNorm: lane = pair, wave w the channels
  // [w chp / 4, (w + 1) chp / 4), in groups of eight (chp <= 256).
  // Channels past ch and pairs past the last repeat one that is there (the
  // pairs are not stored, the channels are zeroed against `live`). The empty
  // asm keeps one pointer and one bound in vector registers: 64 of either would
  // not fit the scalar ones.
  const int groups = a.chp / 32, cw = wave * (a.chp / 4);
  float x[8][8];
  const float* xp = X + (int64_t)min(cw, a.ch - 1) * a.bstride + min(q0 + lane, a.pairs - 1);
  int live = a.ch - cw;
  asm("" : "+v"(live));
#pragma unroll
  for (int i = 0; i < 8; i++) {
    if (i < groups) {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float w = *xp;
        xp += cw + 8 * i + e + 1 < a.ch ? a.bstride : 0;
        asm("" : "+v"(xp));
        x[i][e] = 8 * i + e < live ? w : 0.0f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) x[i][e] = 0.0f;
    }
  }
  {
    const int q = tid >> 2;
    pair_normalize_row<ZT, kMaxSteps>(q0 + q < a.pairs ? z + (int64_t)(a.pair0 + q0 + q) * a.cz : nullptr, a.cz, zsteps, a.eps,
                           a.x_scale, tid & 3, vec, zn + q * zpitch);
  }
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int e = 0; e < 8; e++) s += x[i][e];
  red[wave * 64 + lane] = s;
  __syncthreads();
  const float mean = ((red[lane] + red[64 + lane]) + (red[128 + lane] + red[192 + lane])) / (float)a.ch;
  float d2 = 0.0f;
  const int lives = min(live, 8 * groups);
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      x[i][e] = 8 * i + e < lives ? x[i][e] - mean : 0.0f;
      d2 += x[i][e] * x[i][e];
    }
  red[256 + wave * 64 + lane] = d2;
  __syncthreads();
  d2 = (red[256 + lane] + red[320 + lane]) + (red[384 + lane] + red[448 + lane]);
  const float rstd = fast_rsqrt(d2 / (float)a.ch + a.eps) * a.h_scale;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    if (i >= groups) continue;
    half8 h, l;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      half2v h2, l2;
      pair_split2(x[i][e] * rstd, x[i][e + 1] * rstd, h2, l2);
      h[e] = h2[0], h[e + 1] = h2[1], l[e] = l2[0], l[e + 1] = l2[1];
    }
    half_t* p = hn + lane * hpitch + pair_index(cw + 8 * i);
    *reinterpret_cast<half8*>(p) = h;
    *reinterpret_cast<half8*>(p + 16) = l;
  }
  __syncthreads();

  const half_t* xr = (gate ? zn + (rw + (lane & 31)) * zpitch : hn + (rw + (lane & 31)) * hpitch) + 8 * (lane >> 5);
  float* gates = red + (wave & 1) * 1024;
  OT* out = reinterpret_cast<OT*>(a.out);
  for (int nb = blockIdx.y; nb < blocks; nb += gridDim.y) {
    floatx16 acc = {};
    for (int k = 0; k < steps; k += 2) {
      const PairFragments c = f;
      const int nk = k + 2 < steps ? k + 2 : 0, nn = min(k + 2 < steps ? nb : nb + (int)gridDim.y, blocks - 1);
      f.load(W + nn * block, nk);
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const half8 xh = *reinterpret_cast<const half8*>(xr + 32 * (k + u));
        const half8 xl = *reinterpret_cast<const half8*>(xr + 32 * (k + u) + 16);
        acc = mfma_f16(xh, c.h[u], acc);
        acc = mfma_f16(xh, c.l[u], acc);
        acc = mfma_f16(xl, c.h[u], acc);
      }
    }
    const int n = 32 * nb + (lane & 31);
    const float sc = (gate ? a.s_g : a.s_z)[n], bi = (gate ? a.b_g : a.b_z)[n];
    if (gate) {
#pragma unroll
      for (int v = 0; v < 16; v++) gates[v * 64 + lane] = sigmoidf_(fmaf(acc[v], sc, bi));
    }
    __syncthreads();
    if (!gate) {
      float y[16];
#pragma unroll
      for (int v = 0; v < 16; v++) y[v] = fmaf(acc[v], sc, bi) * gates[v * 64 + lane];
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int q = q0 + rw + mfma_row(v, lane);
        if (n < a.cz && q < a.pairs) {
          const int64_t at = (int64_t)(a.pair0 + q) * a.cz + n;
          out[at] = (OT)(a.residual ? y[v] + (float)out[at] : y[v]);
        }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Weight preparation: f32 [out][in] tensors -> padded CT matrices
// ---------------------------------------------------------------------------

// The fast path's weights with the LayerNorm affines folded in, so its
// kernels normalise to x_hat = (x - mean) / sigma and nothing more:
//   W' = s W diag(gamma),  b' = s (b + W beta),
// gamma, beta the LayerNorm feeding the matrix and s = -log2(e) for the two
// gates (their sigmoid then reads 1 / (1 + 2^acc)). Matrices, in order:
// AP, AG, BP, BG (LayerNorm-in), Z (LayerNorm-out), G (LayerNorm-in), each
// 128 x 128 in MFMA fragment order (fold_index); every product and the bias
// sum are taken in double and rounded once (weights to f16, biases to f32).
struct FoldSources {
  const float* w[kFoldMatrices];
  const float* b[kFoldMatrices];
  const float* gamma[kFoldMatrices];
  const float* beta[kFoldMatrices];
  float scale[kFoldMatrices];
};

__global__ void fold_weights_kernel(FoldSources src, int n_out, int n_in, half_t* __restrict__ w_out,
                                    float* __restrict__ b_out) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= kFoldMatrices * n_out) return;
  const int m = id / n_out, n = id - m * n_out;
  const double s = src.scale[m];
  const float* w = src.w[m] + (size_t)n * n_in;
  double bias = src.b[m][n];
  for (int k = 0; k < n_in; k++) {
    bias += (double)w[k] * (double)src.beta[m][k];
    w_out[fold_index(m, n, k)] = (half_t)(s * (double)w[k] * (double)src.gamma[m][k]);
  }
  b_out[(size_t)m * n_out + n] = (float)(s * bias);
}

template <typename CT>
__global__ void pad_matrix_kernel(const float* __restrict__ src, int rows, int cols, CT* __restrict__ dst,
                                  int prow, int pcol) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)prow * pcol) return;
  int r = (int)(i / pcol), c = (int)(i % pcol);
  dst[i] = (r < rows && c < cols) ? (CT)src[(int64_t)r * cols + c] : (CT)0.0f;
}

__global__ void pad_vector_kernel(const float* __restrict__ src, int n, float* __restrict__ dst, int pn) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < pn) dst[i] = i < n ? src[i] : 0.0f;
}

template <typename CT>
int pad_matrix(const float* src, int rows, int cols, void* dst, int prow, int pcol, hipStream_t s) {
  int64_t n = (int64_t)prow * pcol;
  return launch("tri_prepare", pad_matrix_kernel<CT>, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, s, src, rows,
                cols, (CT*)dst, prow, pcol);
}

int pad_vector(const float* src, int n, void* dst, int pn, hipStream_t s) {
  return launch("tri_prepare", pad_vector_kernel, dim3((unsigned)ceil_div(pn, 256)), dim3(256), 0, s, src, n,
                (float*)dst, pn);
}

int validate(const afhip_triangle_desc* d) {
  AFHIP_REQUIRE(d != nullptr, "descriptor is NULL");
  AFHIP_REQUIRE(d->length > 0 && d->c_z > 0 && d->c_hidden > 0,
                "length, cZ and cHidden must be positive (received %d, %d, %d)", d->length, d->c_z, d->c_hidden);
  AFHIP_REQUIRE((int64_t)d->length * d->length <= (int64_t)1 << 30, "length %d is too large", d->length);
  AFHIP_REQUIRE(d->c_z <= 128, "cZ %d exceeds the 128 channels the output kernel tiles", d->c_z);
  AFHIP_REQUIRE(d->c_hidden <= 256, "cHidden %d exceeds 256", d->c_hidden);
  AFHIP_REQUIRE(d->direction == AFHIP_TRIANGLE_OUTGOING || d->direction == AFHIP_TRIANGLE_INCOMING,
                "unknown direction %d", d->direction);
  AFHIP_REQUIRE(valid_precision(d->precision), "unknown precision %d", d->precision);
  AFHIP_REQUIRE(valid_float_dtype(d->pair_dtype) && valid_float_dtype(d->out_dtype), "pair and output dtypes must be f32 or f16");
  AFHIP_REQUIRE(d->block_rows >= 0, "blockRows must be non-negative");
  AFHIP_REQUIRE(d->epsilon > 0.0f && std::isfinite(d->epsilon), "epsilon must be finite and positive; received %g",
                (double)d->epsilon);
  return AFHIP_OK;
}

template <typename ZT, bool F16MATH>
int launch_project(const ProjectArgs& pa, size_t shared, hipStream_t s) {
  if (int st = allow_lds((const void*)tri_project_kernel<ZT, F16MATH>, shared)) return st;
  return launch("triangle.project", tri_project_kernel<ZT, F16MATH>, dim3((unsigned)ceil_div(pa.P, kRows)),
                dim3(256), shared, s, pa);
}

template <typename ZT, typename OT, bool F16MATH>
int launch_output(const OutputArgs& oa, size_t shared, hipStream_t s) {
  if (int st = allow_lds((const void*)tri_output_kernel<ZT, OT, F16MATH>, shared)) return st;
  return launch("triangle.output", tri_output_kernel<ZT, OT, F16MATH>, dim3((unsigned)ceil_div(oa.pairs, kRows)),
                dim3(256), shared, s, oa);
}

// How many workgroups share a tile's column blocks: enough for two a CU, as
// each of them normalises the tile for itself.
unsigned column_splits(int64_t tiles, int blocks) {
  const int64_t cus = device_cu_count() > 0 ? device_cu_count() : 256;
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(blocks, 2 * cus / tiles));
}

template <typename ZT> int launch_project_pair(const ProjectArgs& pa, hipStream_t s) {
  const int64_t tiles = ceil_div(pa.P, kPairRows);
  const size_t shared = (size_t)kPairRows * pair_pitch(pa.czp / 16) * 2;
  auto k = tri_project_pair_kernel<ZT>;
  if (int st = allow_lds((const void*)k, shared)) return st;
  return launch("triangle.project", k, dim3((unsigned)tiles, column_splits(tiles, pa.chp / 32)), dim3(256), shared, s, pa,
                (int)rows_on_four(pa.z, pa.cz, sizeof(ZT)));
}

// In place one workgroup takes a tile's columns: every workgroup of a tile reads
// all channels of its rows of z for the gate, and nothing orders those reads
// before another one's stores of the same rows.
template <typename ZT, typename OT> int launch_output_pair(const OutputArgs& oa, hipStream_t s) {
  const int64_t tiles = ceil_div(oa.pairs, kPairRows);
  const unsigned splits = oa.in_place ? 1u : column_splits(tiles, (oa.cz + 31) / 32);
  const size_t shared =
      (size_t)kPairRows * (pair_pitch(oa.czp / 16) + pair_pitch(oa.chp / 16)) * 2 + 2 * 32 * 32 * 4;
  auto k = tri_output_pair_kernel<ZT, OT>;
  if (int st = allow_lds((const void*)k, shared)) return st;
  return launch("triangle.output", k, dim3((unsigned)tiles, splits), dim3(256), shared, s, oa,
                (int)rows_on_four(oa.z, oa.cz, sizeof(ZT)));
}

template <bool F16MATH, typename ZT> int launch_output_to(int od, const OutputArgs& oa, size_t shared, hipStream_t s) {
  return od == AFHIP_F32 ? launch_output<ZT, float, F16MATH>(oa, shared, s)
                         : launch_output<ZT, half_t, F16MATH>(oa, shared, s);
}

template <typename ZT> int dispatch_project(Products p, const ProjectArgs& pa, size_t shared, hipStream_t s) {
  if (p == Products::kPairs) return launch_project_pair<ZT>(pa, s);
  return p == Products::kF16 ? launch_project<ZT, true>(pa, shared, s) : launch_project<ZT, false>(pa, shared, s);
}

template <typename ZT> int dispatch_output(Products p, int od, const OutputArgs& oa, size_t shared, hipStream_t s) {
  if (p == Products::kPairs) return od == AFHIP_F32 ? launch_output_pair<ZT, float>(oa, s) : launch_output_pair<ZT, half_t>(oa, s);
  return p == Products::kF16 ? launch_output_to<true, ZT>(od, oa, shared, s)
                             : launch_output_to<false, ZT>(od, oa, shared, s);
}

}  // namespace

}  // namespace afhip

using namespace afhip;

extern "C" {

int afhip_triangle_weights_size(const afhip_triangle_desc* desc, size_t* bytes) {
  if (int s = validate(desc)) return s;
  AFHIP_REQUIRE(bytes != nullptr, "output is NULL");
  *bytes = tri_layout(*desc).total;
  return AFHIP_OK;
}

int afhip_triangle_fast_path(const afhip_triangle_desc* desc, int32_t* fast) {
  if (int s = validate(desc)) return s;
  AFHIP_REQUIRE(fast != nullptr, "output is NULL");
  *fast = triangle_fast_eligible(*desc) ? 1 : 0;
  return AFHIP_OK;
}

int afhip_triangle_workspace_size(const afhip_triangle_desc* desc, size_t* bytes) {
  if (int s = validate(desc)) return s;
  AFHIP_REQUIRE(bytes != nullptr, "output is NULL");
  *bytes = tri_workspace(*desc).total;
  return AFHIP_OK;
}

int afhip_triangle_prepare_weights(const afhip_triangle_desc* desc, const float* packed, void* prepared, void* stream) {
  if (int s = require_open()) return s;
  if (int s = validate(desc)) return s;
  AFHIP_REQUIRE(packed && prepared, "NULL weights");
  const auto& d = *desc;
  const TriWeights w = tri_layout(d);
  hipStream_t st = (hipStream_t)stream;
  const int cz = d.c_z, ch = d.c_hidden;
  // Offsets of the sixteen tensors in ORDER (src/triangle/weights.ts:4-10).
  size_t o[17];
  size_t sizes[16] = {(size_t)cz, (size_t)cz, (size_t)ch * cz, (size_t)ch, (size_t)ch * cz, (size_t)ch,
                      (size_t)ch * cz, (size_t)ch, (size_t)ch * cz, (size_t)ch, (size_t)ch, (size_t)ch,
                      (size_t)cz * ch, (size_t)cz, (size_t)cz * cz, (size_t)cz};
  o[0] = 0;
  for (int i = 0; i < 16; i++) o[i + 1] = o[i] + sizes[i];
  char* base = (char*)prepared;
  if (tri_pairs(d)) {
    // ORDER indices as below; the pair kernels need nothing else.
    PairSources src{};
    auto matrix = [&](int at, int index, int norm, int rows, int cols, int padded, int steps, size_t out, size_t scale,
                      size_t bias) {
      src.m[at] = {packed + o[index], packed + o[index + 1], packed + o[norm], packed + o[norm + 1], rows, cols,
                   padded, steps, pair_norm_exponent(cols), (half_t*)(base + out), (float*)(base + scale),
                   (float*)(base + bias)};
    };
    for (int k = 0; k < 4; k++)
      matrix(k, 2 + 2 * k, 0, ch, cz, w.chp, w.czp / 16, w.w_proj + 4 * (size_t)k * w.chp * w.czp,
             w.s_proj + 4 * (size_t)k * w.chp, w.b_proj + 4 * (size_t)k * w.chp);
    matrix(4, 12, 10, cz, ch, w.czo, w.chp / 16, w.w_z, w.s_z, w.b_z);
    matrix(5, 14, 0, cz, cz, w.czo, w.czp / 16, w.w_g, w.s_g, w.b_g);
    return launch("tri_prepare", tri_pair_prepare_kernel, dim3((unsigned)std::max(w.chp, w.czo), 6), dim3(64), 0, st, src);
  }
  const bool f16 = d.precision == AFHIP_PRECISION_F16;
  const size_t es = f16 ? 2 : 4;
  auto mat = [&](int index, int rows, int cols, size_t dst, int prow, int pcol) {
    return f16 ? pad_matrix<half_t>(packed + o[index], rows, cols, base + dst, prow, pcol, st)
               : pad_matrix<float>(packed + o[index], rows, cols, base + dst, prow, pcol, st);
  };
  int s;
  if ((s = pad_vector(packed + o[0], cz, base + w.ln_in_w, cz, st))) return s;
  if ((s = pad_vector(packed + o[1], cz, base + w.ln_in_b, cz, st))) return s;
  for (int k = 0; k < 4; k++) {  // ap, ag, bp, bg at ORDER 2, 4, 6, 8
    if ((s = mat(2 + 2 * k, ch, cz, w.w_proj + es * (size_t)k * w.chp * w.czp, w.chp, w.czp))) return s;
    if ((s = pad_vector(packed + o[3 + 2 * k], ch, base + w.b_proj + 4 * (size_t)k * w.chp, w.chp, st))) return s;
  }
  if ((s = pad_vector(packed + o[10], ch, base + w.ln_out_w, ch, st))) return s;
  if ((s = pad_vector(packed + o[11], ch, base + w.ln_out_b, ch, st))) return s;
  if ((s = mat(12, cz, ch, w.w_z, w.czo, w.chp))) return s;
  if ((s = pad_vector(packed + o[13], cz, base + w.b_z, w.czo, st))) return s;
  if ((s = mat(14, cz, cz, w.w_g, w.czo, w.czp))) return s;
  if ((s = pad_vector(packed + o[15], cz, base + w.b_g, w.czo, st))) return s;
  if (triangle_fast_eligible(d)) {
    // ORDER indices: LN-in 0/1, AP 2/3, AG 4/5, BP 6/7, BG 8/9, LN-out 10/11, Z 12/13, G 14/15.
    const int wi[kFoldMatrices] = {2, 4, 6, 8, 12, 14};
    const int gi[kFoldMatrices] = {0, 0, 0, 0, 10, 0};
    const float kNegLog2e = -1.4426950408889634f;
    const float sc[kFoldMatrices] = {1.0f, kNegLog2e, 1.0f, kNegLog2e, 1.0f, kNegLog2e};
    FoldSources fs{};
    for (int m = 0; m < kFoldMatrices; m++) {
      fs.w[m] = packed + o[wi[m]];
      fs.b[m] = packed + o[wi[m] + 1];
      fs.gamma[m] = packed + o[gi[m]];
      fs.beta[m] = packed + o[gi[m] + 1];
      fs.scale[m] = sc[m];
    }
    if ((s = launch("tri_prepare", fold_weights_kernel, dim3((unsigned)ceil_div(kFoldMatrices * cz, 128)), dim3(128),
                    0, st, fs, cz, cz, (half_t*)(base + w.fold_w), (float*)(base + w.fold_b))))
      return s;
  }
  return AFHIP_OK;
}

int afhip_triangle_run(const afhip_triangle_desc* desc, const void* z, const float* mask, const void* prepared,
                       void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (int s = require_open()) return s;
  if (int s = validate(desc)) return s;
  AFHIP_REQUIRE(z && mask && prepared && out, "NULL tensor");
  const auto& d = *desc;
  const TriWeights w = tri_layout(d);
  const TriWorkspace ws = tri_workspace(d);
  AFHIP_REQUIRE(workspace != nullptr && workspace_bytes >= ws.total, "workspace of %zu bytes is smaller than %zu",
                workspace_bytes, ws.total);
  hipStream_t st = (hipStream_t)stream;
  const bool f16 = d.precision == AFHIP_PRECISION_F16;
  const Products products = f16 ? Products::kF16 : tri_pairs(d) ? Products::kPairs : Products::kF32;
  const char* wb = (const char*)prepared;
  char* wsb = (char*)workspace;
  const int L = d.length;
  const int P = L * L;

  ProjectArgs pa{};
  pa.z = z;
  pa.mask = mask;
  pa.ln_w = (const float*)(wb + w.ln_in_w);
  pa.ln_b = (const float*)(wb + w.ln_in_b);
  pa.w_proj = wb + w.w_proj;
  pa.b_proj = (const float*)(wb + w.b_proj);
  pa.s_proj = (const float*)(wb + w.s_proj);
  pa.x_scale = ldexpf(1.0f, pair_norm_exponent(d.c_z));
  pa.out_a = wsb + ws.op_a;
  pa.out_b = wsb + ws.op_b;
  pa.cstride = ws.cstride;
  pa.L = L;
  pa.P = P;
  pa.cz = d.c_z;
  pa.ch = d.c_hidden;
  pa.czp = w.czp;
  pa.chp = w.chp;
  pa.incoming = d.direction == AFHIP_TRIANGLE_INCOMING;
  pa.eps = d.epsilon;
  // AlphaFold's widths in f16 take the persistent kernels of
  // triangle_fast.hip; every other shape and the f32 path take the tiles below.
  const bool fast = triangle_fast_eligible(d) && (reinterpret_cast<uintptr_t>(z) & 15) == 0;
  int s;
  if (fast) {
    FastProjectArgs fa{};
    fa.z = z;
    fa.mask = mask;
    fa.w_proj = (const half_t*)(wb + w.fold_w);
    fa.b_proj = (const float*)(wb + w.fold_b);
    fa.out_a = (half_t*)pa.out_a;
    fa.out_b = (half_t*)pa.out_b;
    fa.cstride = ws.cstride;
    fa.L = L;
    fa.P = P;
    fa.incoming = pa.incoming;
    fa.eps = d.epsilon;
    s = launch_triangle_project_f16(fa, d.pair_dtype, st);
  } else {
    const size_t psh = round_up((int64_t)w.czp * (kRows + 1) * 4, 16) +
                       (f16 ? round_up((int64_t)kRows * (w.czp + 8) * 2, 16) : 0) + (size_t)64 * (kRows + 8) * (f16 ? 2 : 4);
    s = d.pair_dtype == AFHIP_F32 ? dispatch_project<float>(products, pa, psh, st)
                                  : dispatch_project<half_t>(products, pa, psh, st);
  }
  if (s) return s;

  // Row operand and column operand of the contraction (see the file comment).
  const void* row_op = pa.incoming ? pa.out_b : pa.out_a;
  const void* col_op = pa.incoming ? pa.out_a : pa.out_b;
  const size_t es = f16 ? 2 : 4;
  GemmTypes types{d.precision, f16 ? AFHIP_F16 : AFHIP_F32, f16 ? AFHIP_F16 : AFHIP_F32, f16 ? AFHIP_F16 : AFHIP_F32};
  const size_t elements = (size_t)P * d.c_z;
  const uintptr_t zb = reinterpret_cast<uintptr_t>(z), ob = reinterpret_cast<uintptr_t>(out);
  const bool in_place = ob < zb + elements * (d.pair_dtype == AFHIP_F16 ? 2 : 4) &&
                        zb < ob + elements * (d.out_dtype == AFHIP_F16 ? 2 : 4);
  const int kmax = std::max(w.chp, w.czp);
  const size_t osh = round_up((int64_t)kmax * (kRows + 1) * 4, 16) + (f16 ? (size_t)kRows * (kmax + 8) * 2 : 0);
  for (int i0 = 0; i0 < L; i0 += ws.block_rows) {
    const int count = std::min(ws.block_rows, L - i0);
    GemmArgs g;
    g.a = (const char*)row_op + es * (size_t)i0 * L;
    g.b = col_op;
    g.c = wsb + ws.contracted;
    g.M = count;
    g.N = L;
    g.K = L;
    g.lda = L;
    g.ldb = L;
    g.ldc = L;
    g.sa = ws.cstride;
    g.sb = ws.cstride;
    g.sc = ws.bstride;
    g.batch = d.c_hidden;
    afhip_variant v = select_variant(types, count, L, L, d.c_hidden);
    if ((s = run_gemm(g, types, v, "triangle.contract", st))) return s;

    OutputArgs oa{};
    oa.contracted = wsb + ws.contracted;
    oa.bstride = ws.bstride;
    oa.z = z;
    oa.ln_in_w = pa.ln_w;
    oa.ln_in_b = pa.ln_b;
    oa.ln_out_w = (const float*)(wb + w.ln_out_w);
    oa.ln_out_b = (const float*)(wb + w.ln_out_b);
    oa.w_z = wb + w.w_z;
    oa.b_z = (const float*)(wb + w.b_z);
    oa.w_g = wb + w.w_g;
    oa.b_g = (const float*)(wb + w.b_g);
    oa.s_z = (const float*)(wb + w.s_z);
    oa.s_g = (const float*)(wb + w.s_g);
    oa.x_scale = pa.x_scale;
    oa.h_scale = ldexpf(1.0f, pair_norm_exponent(d.c_hidden));
    oa.out = out;
    oa.pair0 = i0 * L;
    oa.pairs = count * L;
    oa.cz = d.c_z;
    oa.ch = d.c_hidden;
    oa.czp = w.czp;
    oa.chp = w.chp;
    oa.residual = d.residual;
    oa.in_place = in_place;
    oa.eps = d.epsilon;
    if (fast) {
      FastOutputArgs fo{};
      fo.contracted = (const half_t*)oa.contracted;
      fo.bstride = oa.bstride;
      fo.z = z;
      fo.w_z = (const half_t*)(wb + w.fold_w) + (size_t)4 * kC * kC;
      fo.b_z = (const float*)(wb + w.fold_b) + 4 * kC;
      fo.w_g = (const half_t*)(wb + w.fold_w) + (size_t)5 * kC * kC;
      fo.b_g = (const float*)(wb + w.fold_b) + 5 * kC;
      fo.out = out;
      fo.pair0 = oa.pair0;
      fo.pairs = oa.pairs;
      fo.residual = oa.residual;
      fo.eps = d.epsilon;
      s = launch_triangle_output_f16(fo, d.pair_dtype, d.out_dtype, st);
    } else {
      s = d.pair_dtype == AFHIP_F32 ? dispatch_output<float>(products, d.out_dtype, oa, osh, st)
                                    : dispatch_output<half_t>(products, d.out_dtype, oa, osh, st);
    }
    if (s) return s;
  }
  return AFHIP_OK;
}

}  // extern "C"
