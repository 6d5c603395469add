// Products of a few rows (generation steps): C[m, n] = sum_k A[m, k] B[n, k] for
// M <= kSkinnyRows, where reading B (the weights) once is all the work there is.
#pragma once

#include "cdx_common.h"

namespace cdx {

// Rows up to which the skinny kernels may replace the tile engine (cdx_gemm.h).
constexpr int kSkinnyRows = 64;

// Rows up to which a product can take its A operand through an RMSNorm.
constexpr int kNormRows = 8;

// Whether a product of M rows and N columns runs faster here.  Past 16 rows every block of
// columns re-reads A from L2, which costs in proportion to row groups x column blocks: the
// line lies at 4 per CU (measured on 256 CUs, K = 2048, here against the tile engine: 32
// rows, 8192 columns 14.8 / 16.7 us, 12288 columns 18.8 / 19.7, 32000 columns 37.4 / 35.4;
// 64 rows, 4096 columns (K = 4096) 21.3 / 28.3, 8192 columns 21.5 / 17.1).
bool skinny_fits(int64_t M, int64_t N);

// kF32 stores the fp32 sums; kResid adds the rounded product to bf16 C (the rounding of a
// separate bf16 add); kAccum adds the fp32 product to bf16 C with one rounding.
enum class SkinnyEpi { kStore, kF32, kBiasClamp, kResid, kAccum };

struct SkinnyParams {
  const uint16_t* a;   // [M][lda], K columns [0, k_split)
  int64_t lda;
  const uint16_t* a2;  // K columns [k_split, K) (row stride lda2, 0 = one row for all)
  int64_t lda2;
  const uint16_t* b;   // [N][ldb], K columns [0, k_split)
  const uint16_t* b2;  // K columns [k_split, K), same row stride
  int64_t ldb;
  int32_t k_split;     // == K without a second source; a multiple of 64
  int32_t M, N, K;     // K a multiple of 64
  void* c;             // bf16 (fp32 for kF32), row stride ldc; columns up to round_up(N, 8) are written
  int64_t ldc;
  const uint16_t* bias;  // kBiasClamp: c = clamp(acc + clamp(bias[n], bias_lo, bias_hi), lo, hi)
  float bias_lo, bias_hi, lo, hi;
  // Not null (kF32, M <= kNormRows): columns [0, k_split) of A are RMSNorm(a) with these
  // weights and eps.
  const uint16_t* norm_w;
  float eps;
};

// For shapes that fit (skinny_fits); operands 16-byte aligned, leading dimensions multiples of 8.
int skinny_gemm(const SkinnyParams& p, SkinnyEpi epi, hipStream_t s, const char* name);

// Both MoE passes for 1 <= T <= kSkinnyRows tokens (arguments as cdx_moe_swiglu_fwd); with
// norm_w (T <= kNormRows) of RMSNorm(x).  x may be `out` itself with norm_w and residual: the
// gate/up pass is done with it before the down pass adds to it.
int skinny_moe(const uint16_t* x, int32_t T, int32_t H, int32_t P, int32_t E, bool shared, const int32_t* perm,
               const int32_t* offsets, const uint16_t* w_gu, const uint16_t* w_down, uint16_t* inter, uint16_t* out,
               bool residual, const uint16_t* norm_w, float eps, hipStream_t s, const char* name);

}  // namespace cdx
