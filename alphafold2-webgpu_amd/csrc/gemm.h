// The shared tiled GEMM, as the other translation units launch it.
#pragma once

#include "internal.h"

namespace afhip {

// One batched GEMM launch: C[b][m][n] = epilogue(sum_k A[b][m][k] * B[b][n][k]).
// A is row-major [M][K] (row stride lda), or [K][M] when a_row_contiguous
// (element (m, k) at k * lda + m); B is [N][K] (row stride ldb), the
// k-contiguous layout every kernel here consumes. C is [M][N] (row stride
// ldc), or [N][M] when c_column_major (element (m, n) at n * ldc + m).
struct GemmArgs {
  const void* a = nullptr;
  const void* b = nullptr;
  void* c = nullptr;
  const void* residual = nullptr;
  const float* scale = nullptr;
  const float* bias = nullptr;
  int M = 0, N = 0, K = 0;
  int64_t lda = 0, ldb = 0, ldc = 0;
  int64_t sa = 0, sb = 0, sc = 0;
  int batch = 1;
  bool a_row_contiguous = false;  // the REGISTER_STAGED and LDS_DMA kernels take it
  bool c_column_major = false;    // the REGISTER_STAGED and LDS_DMA kernels take it
  uint32_t flags = 0;
  int head_cols = 0;  // heads * head_dim, ATTENTION only
  float q_scale = 1.0f;
  // Outer-product-mean contraction epilogue: y /= (eps + count[i][j]) with
  // i = (row0 + m) / c_outer, j = n / c_outer; stored at the [i][j][a][b] layout.
  const float* opm_count = nullptr;
  int opm_outer = 0;
  int opm_length = 0;
  int opm_row0 = 0;
  float opm_eps = 0.0f;
  // The fused contraction + output projection (run_opm_fused) only: the
  // output weights in the order opm_fused_weight_index gives.
  const void* opm_w = nullptr;
};

// Epilogue flags private to the library (beyond the public AFHIP_EPILOGUE_*).
// OPM_CONTRACT: y /= (eps + count[i][j]), stored at [i_local][j][a][b].
// OPM_OUTPUT:   y += bias[col] / (eps + count[opm_row0 + row]) (bias scaled by
//               the pair's 1/(eps + count), outer-product-mean.ts:462-479).
constexpr uint32_t EPILOGUE_OPM_CONTRACT = 1u << 16;
constexpr uint32_t EPILOGUE_OPM_OUTPUT = 1u << 17;

// f32 matrices as pairs of f16 (the pair GEMM, gemm_dma.hip): x = h + l with
// h = f16(x), l = f16(x - h), 22 to 24 bits of x wherever 2^-3 <= |x| <= 65504, and
// within 2^-25 below. The callers hold each row's largest element (or a bound on
// it) in [2^14, 2^15) with power-of-two scales, so an element keeps its bits down
// to 2^-17 of that and is within 2^-39 of it below. A
// row keeps each 16 consecutive k as 16 h, then 16 l (64 bytes); a matrix takes
// the bytes it takes in f32. K is a multiple of 16.
__host__ __device__ inline int64_t pair_index(int64_t k) { return 32 * (k >> 4) + (k & 15); }  // of h; l is 16 on
// The empty asm keeps x a rounded f32: contracted into the conversion
// (v_fma_mixlo_f16), the operation that made x would round h from its exact
// result in one place and from x in another, and l would belong to another h.
__device__ __forceinline__ void pair_split(float x, half_t& h, half_t& l) {
  asm("" : "+v"(x));
  h = (half_t)x;
  l = (half_t)(x - (float)h);
}
// Two values at once (v_cvt_pk_f16_f32).
__device__ __forceinline__ void pair_split2(float x0, float x1, half2v& h, half2v& l) {
  typedef float float2v __attribute__((ext_vector_type(2)));
  asm("" : "+v"(x0), "+v"(x1));
  h = __builtin_convertvector(float2v{x0, x1}, half2v);
  // v_fma_mix_f32 reads h as it is
  const float d0 = __builtin_fmaf((float)h[0], -1.0f, x0), d1 = __builtin_fmaf((float)h[1], -1.0f, x1);
  l = __builtin_convertvector(float2v{d0, d1}, half2v);
}
__device__ __forceinline__ void pair_store(half_t* row, int64_t k, float x) {
  half_t h, l;
  pair_split(x, h, l);
  row[pair_index(k)] = h;
  row[pair_index(k) + 16] = l;
}
// The power of two (its exponent) that takes values of magnitude up to `most`
// into [-2^15, 2^15], the largest past 2^14; 0 where there are none. An infinite
// `most` is a bound past the largest f32 on values that are none of them past it.
__device__ __forceinline__ int pair_exponent_of(float most) {
  if (!(most > 0.0f)) return 0;
  int p;
  frexpf(fminf(most, 3.402823466e38f), &p);  // m 2^p, m in [1/2, 1)
  return 15 - p;
}
// Bounded so that the exponents a result adds up stay in f32.
__device__ __forceinline__ int pair_exponent(float most) { return min(pair_exponent_of(most), 110); }
// A LayerNorm's output before its affine: C values of magnitude at most
// sqrt(C), stored times 2^pair_norm_exponent(C), at most 2^15.
inline int pair_norm_exponent(int C) {
  int root = 0;
  while ((int64_t)1 << (2 * root) < C) root++;  // sqrt(C) <= 2^root
  return 15 - root;
}
// Below this many products a sum stays on the f32 MFMA. The pairs keep 22 to 24
// bits of an operand and drop the l l term (2^-24 of a product), but a third as
// many f32 roundings accumulate, which is worth less the shorter the sum.
// Measured against 64 bits, operators over pairs / on the f32 MFMA (rms error):
// transition 16 x 16 1.30, 32 x 32 1.15, 64 x 64 0.99, 256 x 1024 0.83; triangle
// 16 x 16 1.13, 32 x 32 1.02, 64 x 64 0.91; attention over 20 keys, 16 channels
// 1.16, 32 1.05, 64 0.93, 256 0.74; outer-product mean 16 channels 1.06, 64 0.99.
constexpr int kPairMinK = 64;
// The output as pairs (rows of ldc elements, 2 ldc halves) instead of TC.
constexpr uint32_t EPILOGUE_PAIRS = 1u << 18;

// C = epilogue(sum_k (A_h B_h + A_h B_l + A_l B_h)) over pair rows: A [M], B [N]
// rows of K elements, f32 accumulation, epilogue SCALE, BIAS, ATTENTION (the
// gate's sigmoid; q as it is), RELU and RESIDUAL (f32 or f16 outputs only) in
// that order. N, ldc and head_cols multiples of 16, operands on 4 bytes (16 for
// the wide loads), no batch, K at least kPairMinK.
int run_gemm_pairs(const GemmArgs& args, int c_dtype, const char* label, hipStream_t stream);

struct GemmTypes {
  int precision;  // AFHIP_PRECISION_*
  int a_dtype;    // AFHIP_F32 | AFHIP_F16
  int b_dtype;    // AFHIP_F32 | AFHIP_F16 | AFHIP_I8
  int c_dtype;    // AFHIP_F32 | AFHIP_F16
};

// Runs one GEMM with the given variant (tile shape); the variant's
// vectorized flag is ignored and derived from alignment.
int run_gemm(const GemmArgs& args, const GemmTypes& types, const afhip_variant& variant, const char* label,
             hipStream_t stream);

// Heuristic kernel and tile choice for a problem of these types and size.
afhip_variant heuristic_variant(const GemmTypes& types, int64_t M, int64_t N, int64_t K, int batch);
// The REGISTER_STAGED variant for a shape: what takes every operand form.
afhip_variant register_variant(int precision, int64_t M, int64_t N, int64_t K, int batch);

// The LDS_DMA kernel family (gemm_dma.hip): f16 arithmetic on an f16 or f32
// A and an f16 B (k-contiguous), or f32 arithmetic on f32 operands.
bool dma_tile_supported(int tile_m, int tile_n);
bool dma_eligible(const GemmArgs& args, const GemmTypes& types);
void dma_heuristic_tile(int64_t M, int64_t N, int64_t K, int64_t batch, int* tile_m, int* tile_n);
int run_gemm_dma(const GemmArgs& args, const GemmTypes& types, int tile_m, int tile_n, const char* label,
                 hipStream_t stream);

// The outer-product mean's contraction and output projection in one launch
// (gemm_dma.hip), for f16 arithmetic with c_outer = 32 and c_z in (96, 128]:
// A = left [L * 32][K], B = right [L * 32][K] (rows i * 32 + a, k-contiguous,
// row stride lda = ldb), count [L][L], opm_w the permuted output weights,
// bias [128], out [L][L][c_z] (row stride ldc = c_z) of dtype c_dtype, plus
// the old contents when flags has AFHIP_EPILOGUE_RESIDUAL. Every pair (i, j)
// computes
//   outer[a][b] = f16(sum_s left[i * 32 + a][s] right[j * 32 + b][s] / (eps + count[i][j]))
//   out[i][j][z] = sum_(a, b) outer[a][b] W[a * 32 + b][z] + bias[z] / (eps + count[i][j]).
int run_opm_fused(const GemmArgs& args, int c_dtype, const char* label, hipStream_t stream);
// Where W[k][z] (k = a * 32 + b, z < 128) sits in the fused kernel's
// 128 x 1024 f16 weight array. The pair rows in LDS hold (a, b) at half
// k' = 128 (b / 4) + 4 a + b % 4; an MFMA step reads 16-byte chunk
// c = 8 Q + 4 h + t of a row (k' in [8 c, 8 c + 8)) in lane half h, so the
// array is stored in the order the lanes load it, [z / 32][Q][t][h][z % 32]
// [k' % 8]: every wave-level load of a step's B fragment is 1 KiB contiguous.
__host__ __device__ inline int64_t opm_fused_weight_index(int k, int z) {
  const int a = k >> 5, b = k & 31;
  const int kp = 128 * (b >> 2) + 4 * a + (b & 3);
  const int c = kp >> 3, Q = c >> 3, h = (c >> 2) & 1, t = c & 3;
  return (((((int64_t)(z >> 5) * 16 + Q) * 4 + t) * 2 + h) * 32 + (z & 31)) * 8 + (kp & 7);
}

// The STREAM kernel (gemm_stream.hip): f16 activations and output, f16 or
// int8 weights held in registers, K in {64, 128, 256}, N % 64 == 0.
bool stream_shape_ok(const GemmTypes& types, int64_t M, int64_t N, int64_t K, int batch);
bool stream_eligible(const GemmArgs& args, const GemmTypes& types);
// add_f16: out += f16(result) in f32 with one more rounding (the attention
// output's residual), after a plain bias epilogue, at K <= 128.
int run_gemm_stream(const GemmArgs& args, const GemmTypes& types, const char* label, hipStream_t stream,
                    bool add_f16 = false);

// The variant plans of this shape should use (pinned, calibrated or heuristic).
afhip_variant select_variant(const GemmTypes& types, int64_t M, int64_t N, int64_t K, int batch);
// select_variant for a whole description: its layouts, strides and the
// weight dtype the kernels read included (types as the description gives
// them).
afhip_variant select_plan_variant(const afhip_gemm_desc& desc, const GemmTypes& types);

// W[k][n] (src) -> W[n][k] (dst), with dtype conversion.
int pack_transpose(const void* src, int src_dtype, int rows_k, int cols_n, int64_t ld_src, void* dst,
                   int dst_dtype, int64_t ld_dst, hipStream_t stream);

// afhip_gemm_run after its open check: `workspace` holds the plan's
// afhip_gemm_workspace_size bytes (or more) when the plan needs any.
int run_gemm_plan(const afhip_gemm_plan* plan, const void* a, const void* w, const float* scale, const float* bias,
                  const void* residual, void* c, void* workspace, size_t workspace_bytes, void* stream);

// Elementwise f32 -> dst dtype conversion (dst may be F32: plain copy).
int convert_f32(const float* src, int64_t count, void* dst, int dst_dtype, hipStream_t stream);

}  // namespace afhip
