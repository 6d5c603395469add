// Attention of a generation for gfx950: QK RMSNorm, RoPE and the KV cache after a plain
// mu-QKV product, and the V^T layout of a cache for the attention kernel.
//
// Reference behaviour: core/attention.py:138-175 (per-head QK norm, RoPE at positions
// past .. past + S - 1, k and v appended to the cache, causal attention whose mask is
// aligned at the top left: query i of the call sees keys 0 .. i of the whole cache).
//
//   qkv_cache_kernel  reads the packed projection [M][(nq + 2 nkv) D] once.  16 lanes hold
//                     one head of one token (lane i columns 4 i .. 4 i + 3 of each half,
//                     so both elements of every RoPE pair), which covers any head
//                     dimension up to 128 that is a multiple of 8.  K and V rows go to row
//                     past + s of the new cache; further blocks copy the old cache there,
//                     16 bytes per lane.  The work is one pass over the cache, which is
//                     what bounds a step.  With few queries whose keys all lie in the old
//                     cache (S <= kAttendRows, past >= S) a query's 16 lanes also run its
//                     attention, so a step needs no further launch.
//                     Measured with the product (us): 4 sequences of 1000 cached tokens,
//                     8 KV heads of 128 (33 MB through the cache) 14.5, of which the
//                     product 8; 1 sequence of 500, 4 KV heads of 64: 6.7.
//   vt_pack_kernel    [rows][D] -> V^T tiles in the key order of the attention kernel
//                     (2 x 777 tokens, 4 heads of 80: 3.6 us; a prompt's own V^T is written by
//                     the pass above instead).
#include "cdx_gemm.h"
#include "cdx_skinny.h"

namespace cdx {
namespace {

constexpr int kAttendRows = 16;
constexpr int kCopyVec = 4;  // 16-byte pieces a lane copies

struct QkvCacheParams {
  const void* qkv;  // [M][(nq + 2 nkv) D], fp32 or bf16
  int32_t B, S, nq, nkv, D;
  const uint16_t* q_norm_w;  // [D], nullptr = no QK norm
  const uint16_t* k_norm_w;
  float eps;
  const float* cos_sin;  // [pos][D / 2][2]
  int32_t past;          // rows of the old cache = position of token 0
  const uint16_t* past_k;  // [B][nkv][past][D]
  const uint16_t* past_v;
  uint16_t* q;  // [B][nq][S][D], or nullptr: attend
  uint16_t* k;  // [B][nkv][past + S][D]
  uint16_t* v;
  uint16_t* attn;  // [B][S][nq D]
  float scale_log2;
  uint16_t* vt;         // V^T of the new tokens (past == 0), [B][nkv][D][vt_ld], or nullptr
  int64_t vt_ld;
  uint32_t row_blocks;  // blocks of 16 (token, head) rows; those after them copy, or write V
};

// Sum over each row of 16 lanes, returned to all of them.
__device__ __forceinline__ float row16_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, false));
  return v;
}

__device__ __forceinline__ void load4(const float* p, float* f) {
  const float4 v = *reinterpret_cast<const float4*>(p);
  f[0] = v.x, f[1] = v.y, f[2] = v.z, f[3] = v.w;
}
__device__ __forceinline__ void load4(const uint16_t* p, float* f) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  f[0] = __uint_as_float(v.x << 16), f[1] = __uint_as_float(v.x & 0xffff0000u);
  f[2] = __uint_as_float(v.y << 16), f[3] = __uint_as_float(v.y & 0xffff0000u);
}
__device__ __forceinline__ void store4(uint16_t* p, const float* f) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]));
}

// A staged tile of 64 tokens x D values in LDS (rows of D + 8) to columns s0 .. s0 + 63 of
// V^T rows (vt_ld apart) in vt_col order: 16-byte writes along the tokens.
__device__ __forceinline__ void store_vt_tile(const uint16_t* tile, int D, uint16_t* dst, int64_t vt_ld) {
  const int pitch = D + 8;
  for (int i = threadIdx.x; i < D * 8; i += 256) {
    const int d = i >> 3, ck = i & 7;
    // Columns 8 ck .. 8 ck + 7 hold tokens t .. t + 3 and t + 8 .. t + 11 (vt_col).
    const uint16_t* p = tile + (16 * (ck >> 1) + 4 * (ck & 1)) * pitch + d;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = (j >> 1) * 8 + (j & 1) * 2;
      w[j] = (uint32_t)p[t * pitch] | ((uint32_t)p[(t + 1) * pitch] << 16);
    }
    *reinterpret_cast<uint4*>(dst + (int64_t)d * vt_ld + ck * 8) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

__device__ __forceinline__ uint4 load8_bf16(const float* p) {
  float f[8];
  load4(p, f);
  load4(p + 4, f + 4);
  return pack8(f);
}
__device__ __forceinline__ uint4 load8_bf16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }

// VT: the V heads go by blocks of 64 tokens, which write the cache rows and, through LDS, V^T
// for the attention kernel (no pass of its own over V).
template <typename TIn, bool VT>
__global__ __launch_bounds__(256) void qkv_cache_kernel(const QkvCacheParams p) {
  const int rows_out = p.past + p.S;
  if (VT && blockIdx.x >= p.row_blocks) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[VT ? 64 * (128 + 8) : 8];
    const uint32_t vb = blockIdx.x - p.row_blocks, tiles = (p.S + 63) / 64;
    const uint32_t slab = vb / tiles;
    const int s0 = (int)(vb - slab * tiles) * 64, b = slab / p.nkv, h = slab - b * p.nkv;
    const int cpr = p.D / 8, heads = p.nq + 2 * p.nkv;
    for (int i = threadIdx.x; i < 64 * cpr; i += 256) {
      const int t = i / cpr, ch = i - t * cpr;
      uint4 x = make_uint4(0u, 0u, 0u, 0u);
      if (s0 + t < p.S) {
        const int64_t m = (int64_t)b * p.S + s0 + t;
        x = load8_bf16(static_cast<const TIn*>(p.qkv) + (m * heads + p.nq + p.nkv + h) * p.D + ch * 8);
        *reinterpret_cast<uint4*>(p.v + ((int64_t)slab * rows_out + s0 + t) * p.D + ch * 8) = x;
      }
      *reinterpret_cast<uint4*>(tile + t * (p.D + 8) + ch * 8) = x;
    }
    __syncthreads();
    store_vt_tile(tile, p.D, p.vt + (int64_t)slab * p.D * p.vt_ld + s0, p.vt_ld);
    return;
  }
  if (!VT && blockIdx.x >= p.row_blocks) {
    // The old cache: slab (b, kv head) of past * D values moves to slab stride
    // (past + S) * D; K slabs, then V slabs.  (The host bounds the counts to 31 bits.)
    const uint32_t slab = (uint32_t)p.past * p.D / 8, n = slab * p.B * p.nkv;
    const uint32_t grow = (uint32_t)p.S * p.D / 8;
    const uint32_t i0 = (blockIdx.x - p.row_blocks) * (256 * kCopyVec) + threadIdx.x;
    uint4 x[kCopyVec];
#pragma unroll
    for (int u = 0; u < kCopyVec; ++u) {
      const uint32_t i = min(i0 + u * 256, 2 * n - 1);
      x[u] = reinterpret_cast<const uint4*>(i < n ? p.past_k : p.past_v)[i < n ? i : i - n];
    }
#pragma unroll
    for (int u = 0; u < kCopyVec; ++u) {
      const uint32_t i = i0 + u * 256;
      const uint32_t j = i < n ? i : i - n;
      if (i < 2 * n) store_nt16(reinterpret_cast<uint4*>(i < n ? p.k : p.v) + (j + j / slab * grow), x[u]);
    }
    return;
  }

  const int g16 = threadIdx.x & 15;
  const int heads = p.nq + (VT ? 1 : 2) * p.nkv;  // heads of a token that go by rows
  const int64_t rows = (int64_t)p.B * p.S * heads;
  const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int half = p.D >> 1;
  // Lanes past the head (and groups past the last row) take part in the row sums with
  // zeros and store nothing.
  const bool on = row < rows && 4 * g16 < half;
  const int64_t rr = row < rows ? row : rows - 1;
  const int64_t m = rr / heads;
  const int head = (int)(rr - m * heads);
  const int64_t b = m / p.S;
  const int s = (int)(m - b * p.S);
  const int kind = head < p.nq ? 0 : (head < p.nq + p.nkv ? 1 : 2);
  const int h = kind == 0 ? head : (kind == 1 ? head - p.nq : head - p.nq - p.nkv);
  const int c = on ? 4 * g16 : 0;

  // Every operand is on its way before the first is used: head, norm weights, rotary pairs
  // and, for an attending query, its first key and value.  (V rows load the q weights and
  // their rotary pairs too, unused: no branches between the loads.)
  const bool attend = p.q == nullptr;
  const uint16_t* nw = kind == 1 ? p.k_norm_w : p.q_norm_w;
  const bool norm = nw != nullptr && kind != 2;
  const TIn* src = static_cast<const TIn*>(p.qkv) + (m * (p.nq + 2 * p.nkv) + head) * p.D + c;
  const float* cs = p.cos_sin + ((int64_t)(p.past + s) * half + c) * 2;
  const int64_t base = (b * p.nkv + h / (p.nq / p.nkv)) * p.past * p.D + c;  // the query's old cache slab
  float x1[4], x2[4], t[8], w1[4] = {1.f, 1.f, 1.f, 1.f}, w2[4] = {1.f, 1.f, 1.f, 1.f};
  float k1[4], k2[4], v1[4], v2[4];
  load4(src, x1);
  load4(src + half, x2);
  load4(cs, t);
  load4(cs + 4, t + 4);
  if (nw != nullptr) {
    load4(nw + c, w1);
    load4(nw + c + half, w2);
  }
  if (attend && kind == 0) {
    load4(p.past_k + base, k1);
    load4(p.past_k + base + half, k2);
    load4(p.past_v + base, v1);
    load4(p.past_v + base + half, v2);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (kind != 2) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) ss = __builtin_fmaf(x1[j], x1[j], __builtin_fmaf(x2[j], x2[j], ss));
    const float rs = rsqrtf(row16_sum(on ? ss : 0.f) / (float)p.D + p.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x1[j] = norm ? w1[j] * (x1[j] * rs) : x1[j];
      x2[j] = norm ? w2[j] * (x2[j] * rs) : x2[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = x1[j], z = x2[j];
      x1[j] = __builtin_fmaf(a, t[2 * j], -(z * t[2 * j + 1]));
      x2[j] = __builtin_fmaf(z, t[2 * j], a * t[2 * j + 1]);
    }
  }
  if (kind != 0) {
    if (!on) return;
    uint16_t* dst = (kind == 1 ? p.k : p.v) + ((b * p.nkv + h) * rows_out + p.past + s) * p.D + c;
    store4(dst, x1);
    store4(dst + half, x2);
    return;
  }
  if (!attend) {
    if (!on) return;
    uint16_t* dst = p.q + ((b * p.nq + h) * p.S + s) * p.D + c;
    store4(dst, x1);
    store4(dst + half, x2);
    return;
  }
  // Attention of query s over keys 0 .. s of the old cache (the host has past >= S):
  // online softmax in log2 units, everything in fp32.
  float mx = -INFINITY, l = 0.f, o1[4] = {0.f, 0.f, 0.f, 0.f}, o2[4] = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j <= s; ++j) {
    if (j > 0) {
      const int64_t at = base + (int64_t)j * p.D;
      load4(p.past_k + at, k1);
      load4(p.past_k + at + half, k2);
      load4(p.past_v + at, v1);
      load4(p.past_v + at + half, v2);
    }
    float dot = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) dot = __builtin_fmaf(x1[i], k1[i], __builtin_fmaf(x2[i], k2[i], dot));
    const float z = row16_sum(on ? dot : 0.f) * p.scale_log2;
    // A score of -inf weighs nothing, also as the first (where z - m_new has no value); +inf and
    // NaN make the row NaN, as do scores of -inf alone (l stays 0).
    const float m_new = fmaxf(mx, z);
    const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(mx - m_new);
    const float w = z == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(z - m_new);
    mx = m_new;
    l = l * alpha + w;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o1[i] = __builtin_fmaf(w, v1[i], o1[i] * alpha);
      o2[i] = __builtin_fmaf(w, v2[i], o2[i] * alpha);
    }
  }
  if (!on) return;
  const float inv = 1.f / l;
#pragma unroll
  for (int i = 0; i < 4; ++i) o1[i] *= inv, o2[i] *= inv;
  uint16_t* dst = p.attn + (m * p.nq + h) * p.D + c;
  store4(dst, o1);
  store4(dst + half, o2);
}

// V [slabs][rows][D] (tokens 0 .. S - 1 of each slab) to V^T [slabs][D][vt_ld]: a block
// moves 64 tokens of one slab through LDS, 16-byte reads along D, 16-byte writes along the
// tokens in vt_col order.  Columns of tokens >= S are cleared.  (The slabs are not a grid
// dimension of their own: y and z end at 65535, which batch x heads may exceed.)
__global__ __launch_bounds__(256) void vt_pack_kernel(const uint16_t* __restrict__ v, int64_t rows, int S, int D,
                                                      uint16_t* __restrict__ vt, int64_t vt_ld) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[64 * (128 + 8)];
  const int pitch = D + 8, cpr = D / 8;
  const uint32_t tiles = ((uint32_t)S + 63) / 64, slab = blockIdx.x / tiles;
  const int s0 = (int)(blockIdx.x - slab * tiles) * 64;
  const uint16_t* src = v + ((int64_t)slab * rows + s0) * D;
  for (int i = threadIdx.x; i < 64 * cpr; i += 256) {
    const int t = i / cpr, ch = i - t * cpr;
    uint4 x = make_uint4(0u, 0u, 0u, 0u);
    if (s0 + t < S) x = *reinterpret_cast<const uint4*>(src + (int64_t)t * D + ch * 8);
    *reinterpret_cast<uint4*>(tile + t * pitch + ch * 8) = x;
  }
  __syncthreads();
  store_vt_tile(tile, D, vt + (int64_t)slab * D * vt_ld + s0, vt_ld);
}

}  // namespace
}  // namespace cdx

extern "C" int32_t cdx_few_rows(int64_t M, int64_t N) { return M > 0 && N > 0 && cdx::skinny_fits(M, N) ? 1 : 0; }

extern "C" size_t cdx_qkv_cache_workspace_bytes(int64_t B, int64_t S, int32_t nq, int32_t nkv, int32_t hd) {
  if (B <= 0 || S <= 0 || nq <= 0 || nkv <= 0 || hd <= 0) return 0;
  const int64_t M = B * S, N = ((int64_t)nq + 2 * (int64_t)nkv) * hd;
  return (size_t)(M * N) * (cdx::skinny_fits(M, N) ? sizeof(float) : sizeof(uint16_t));
}

namespace cdx {
namespace {

int qkv_cache(const char* name, const uint16_t* x_norm_w, float x_eps, const uint16_t* x, int64_t ldx,
              const uint16_t* mu, int64_t ldmu, const uint16_t* w, const uint16_t* w_mu, int64_t ldw, int64_t B,
              int64_t S, int32_t H, int32_t nq, int32_t nkv, int32_t hd, const uint16_t* q_norm_w,
              const uint16_t* k_norm_w, float eps, const float* cos_sin, int64_t n_pos, const uint16_t* past_k,
              const uint16_t* past_v, int64_t past, uint16_t* q_out, uint16_t* k_out, uint16_t* v_out,
              uint16_t* attn_out, float scale, void* work, size_t work_bytes, void* stream, uint16_t* vt = nullptr,
              int64_t vt_ld = 0) {
  clear_error();
  if (B < 0 || S < 0 || H <= 0 || nq <= 0 || nkv <= 0 || nq % nkv != 0 || past < 0 || n_pos < 0)
    return fail(CDX_EINVAL, "%s: bad shape B=%lld S=%lld H=%d nq=%d nkv=%d past=%lld", name, (long long)B,
                (long long)S, H, nq, nkv, (long long)past);
  if (hd <= 0 || hd > 128 || hd % 8 != 0)
    return fail(CDX_EUNSUPPORTED, "%s: head dim %d must be a multiple of 8 and <= 128", name, hd);
  if (H % 64 != 0) return fail(CDX_EUNSUPPORTED, "%s: H=%d must be a multiple of 64", name, H);
  if ((q_norm_w == nullptr) != (k_norm_w == nullptr))
    return fail(CDX_EINVAL, "%s: q and k norm weights must both be given or both be NULL", name);
  if (!(eps >= 0.f)) return fail(CDX_EINVAL, "%s: eps must be >= 0", name);
  if ((q_out == nullptr) == (attn_out == nullptr))
    return fail(CDX_EINVAL, "%s: one of q_out and attn_out must be given", name);
  if (attn_out && (S > kAttendRows || past < S))
    return fail(CDX_EUNSUPPORTED, "%s: attn_out needs S <= %d and past >= S", name, kAttendRows);
  if (vt && (past != 0 || attn_out || vt_ld < S || vt_ld % 64 != 0 || !aligned16(vt)))
    return fail(CDX_EINVAL, "%s: vt_out needs past == 0, q_out and vt_ld >= S, a multiple of 64", name);
  if (attn_out && !(scale > 0.f)) return fail(CDX_EINVAL, "%s: scale must be > 0", name);
  if (ldx < H || ldw < H || (mu && ldmu != 0 && ldmu < H))
    return fail(CDX_EINVAL, "%s: leading dimension too small", name);
  if (ldx % 8 || ldw % 8 || (mu && ldmu % 8))
    return fail(CDX_EUNSUPPORTED, "%s: leading dimensions must be multiples of 8", name);
  const int64_t M = B * S, N = ((int64_t)nq + 2 * (int64_t)nkv) * hd;
  if (M == 0) return CDX_OK;
  // The kernel counts 16-byte pieces of both caches, and (token, head) rows, in 32 bits.
  if (N > INT32_MAX || past + S > INT32_MAX || M > INT32_MAX || B * nkv > INT32_MAX ||
      2 * B * nkv * (past + S) > INT32_MAX / (hd / 8) || M > INT32_MAX / (nq + 2 * nkv))
    return fail(CDX_EUNSUPPORTED, "%s: problem too large", name);
  if (past + S > n_pos)
    return fail(CDX_EINVAL, "%s: cos/sin table has %lld positions, needs %lld", name, (long long)n_pos,
                (long long)(past + S));
  if (!x || !w || (mu && !w_mu) || !cos_sin || !k_out || !v_out || !work || (past > 0 && (!past_k || !past_v)))
    return fail(CDX_EINVAL, "%s: null pointer", name);
  if (!aligned16(x) || !aligned16(w) || (mu && (!aligned16(mu) || !aligned16(w_mu))) || !aligned16(cos_sin) ||
      !aligned16(k_out) || !aligned16(v_out) || !aligned16(work) || !aligned16(past_k) || !aligned16(past_v) ||
      !aligned16(q_out) || !aligned16(attn_out) || !aligned16(q_norm_w) || !aligned16(k_norm_w))
    return fail(CDX_EUNSUPPORTED, "%s: pointers must be 16-byte aligned", name);
  const size_t need = cdx_qkv_cache_workspace_bytes(B, S, nq, nkv, hd);
  if (work_bytes < need)
    return fail(CDX_EWORKSPACE, "%s: workspace needs %zu bytes, got %zu", name, need, work_bytes);

  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool few = skinny_fits(M, N);
  if (x_norm_w && (!few || M > kNormRows))
    return fail(CDX_EUNSUPPORTED, "%s: a folded norm needs B * S <= %d", name, kNormRows);
  if (few) {
    SkinnyParams sp{};
    sp.a = x;
    sp.lda = ldx;
    sp.a2 = mu ? mu : x;
    sp.lda2 = mu ? ldmu : ldx;
    sp.b = w;
    sp.b2 = mu ? w_mu : w;
    sp.ldb = ldw;
    sp.k_split = H;
    sp.M = (int32_t)M;
    sp.N = (int32_t)N;
    sp.K = mu ? 2 * H : H;
    sp.c = work;
    sp.ldc = N;
    sp.norm_w = x_norm_w;
    sp.eps = x_eps;
    if (int rc = skinny_gemm(sp, SkinnyEpi::kF32, s, name)) return rc;
  } else if (int rc = cdx_mu_qkv_fwd(x, ldx, mu, ldmu, w, w_mu, ldw, M, H, (int32_t)N, static_cast<uint16_t*>(work), N,
                                     stream)) {
    return rc;
  }
  QkvCacheParams p{};
  p.qkv = work;
  p.B = (int32_t)B;
  p.S = (int32_t)S;
  p.nq = nq;
  p.nkv = nkv;
  p.D = hd;
  p.q_norm_w = q_norm_w;
  p.k_norm_w = k_norm_w;
  p.eps = eps;
  p.cos_sin = cos_sin;
  p.past = (int32_t)past;
  p.past_k = past_k;
  p.past_v = past_v;
  p.q = q_out;
  p.k = k_out;
  p.v = v_out;
  p.attn = attn_out;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.vt = vt;
  p.vt_ld = vt_ld;
  p.row_blocks = (uint32_t)((M * (nq + (vt ? 1 : 2) * nkv) + 15) / 16);
  if (vt) {
    const dim3 grid(p.row_blocks + (uint32_t)((S + 63) / 64 * B * nkv));
    if (few)
      qkv_cache_kernel<float, true><<<grid, dim3(256), 0, s>>>(p);
    else
      qkv_cache_kernel<uint16_t, true><<<grid, dim3(256), 0, s>>>(p);
    return check_launch(name);
  }
  const int64_t copies = 2 * B * nkv * past * hd / 8;
  const dim3 grid(p.row_blocks + (uint32_t)((copies + 256 * kCopyVec - 1) / (256 * kCopyVec)));
  if (few)
    qkv_cache_kernel<float, false><<<grid, dim3(256), 0, s>>>(p);
  else
    qkv_cache_kernel<uint16_t, false><<<grid, dim3(256), 0, s>>>(p);
  return check_launch(name);
}

}  // namespace
}  // namespace cdx

extern "C" int cdx_qkv_cache_fwd(const uint16_t* x, int64_t ldx, const uint16_t* mu, int64_t ldmu, const uint16_t* w,
                                 const uint16_t* w_mu, int64_t ldw, int64_t B, int64_t S, int32_t H, int32_t nq,
                                 int32_t nkv, int32_t hd, const uint16_t* q_norm_w, const uint16_t* k_norm_w,
                                 float eps, const float* cos_sin, int64_t n_pos, const uint16_t* past_k,
                                 const uint16_t* past_v, int64_t past, uint16_t* q_out, uint16_t* k_out,
                                 uint16_t* v_out, uint16_t* attn_out, float scale, void* work, size_t work_bytes,
                                 void* stream) {
  return cdx::qkv_cache("cdx_qkv_cache_fwd", nullptr, 0.f, x, ldx, mu, ldmu, w, w_mu, ldw, B, S, H, nq, nkv, hd,
                        q_norm_w, k_norm_w, eps, cos_sin, n_pos, past_k, past_v, past, q_out, k_out, v_out, attn_out,
                        scale, work, work_bytes, stream);
}

extern "C" int cdx_qkv_prompt_fwd(const uint16_t* x, int64_t ldx, const uint16_t* mu, int64_t ldmu, const uint16_t* w,
                                  const uint16_t* w_mu, int64_t ldw, int64_t B, int64_t S, int32_t H, int32_t nq,
                                  int32_t nkv, int32_t hd, const uint16_t* q_norm_w, const uint16_t* k_norm_w,
                                  float eps, const float* cos_sin, int64_t n_pos, uint16_t* q_out, uint16_t* k_out,
                                  uint16_t* v_out, uint16_t* vt_out, int64_t vt_ld, void* work, size_t work_bytes,
                                  void* stream) {
  using namespace cdx;
  clear_error();
  const char* name = "cdx_qkv_prompt_fwd";
  if (!vt_out) return fail(CDX_EINVAL, "%s: null pointer", name);
  return qkv_cache(name, nullptr, 0.f, x, ldx, mu, ldmu, w, w_mu, ldw, B, S, H, nq, nkv, hd, q_norm_w, k_norm_w, eps,
                   cos_sin, n_pos, nullptr, nullptr, 0, q_out, k_out, v_out, nullptr, 1.f, work, work_bytes, stream,
                   vt_out, vt_ld);
}

extern "C" int cdx_qkv_cache_norm_fwd(const uint16_t* h, int64_t ldh, const uint16_t* norm_w, float norm_eps,
                                      const uint16_t* mu, int64_t ldmu, const uint16_t* w, const uint16_t* w_mu,
                                      int64_t ldw, int64_t B, int64_t S, int32_t H, int32_t nq, int32_t nkv,
                                      int32_t hd, const uint16_t* q_norm_w, const uint16_t* k_norm_w, float eps,
                                      const float* cos_sin, int64_t n_pos, const uint16_t* past_k,
                                      const uint16_t* past_v, int64_t past, uint16_t* q_out, uint16_t* k_out,
                                      uint16_t* v_out, uint16_t* attn_out, float scale, void* work,
                                      size_t work_bytes, void* stream) {
  using namespace cdx;
  const char* name = "cdx_qkv_cache_norm_fwd";
  clear_error();
  if (!norm_w || !aligned16(norm_w)) return fail(CDX_EINVAL, "%s: bad norm weight pointer", name);
  if (!(norm_eps >= 0.f)) return fail(CDX_EINVAL, "%s: eps must be >= 0", name);
  return qkv_cache(name, norm_w, norm_eps, h, ldh, mu, ldmu, w, w_mu, ldw, B, S, H, nq, nkv, hd, q_norm_w, k_norm_w,
                   eps, cos_sin, n_pos, past_k, past_v, past, q_out, k_out, v_out, attn_out, scale, work, work_bytes,
                   stream);
}

extern "C" int cdx_vt_pack(const uint16_t* v, int64_t slabs, int64_t rows, int64_t S, int32_t hd, uint16_t* vt,
                           int64_t vt_ld, void* stream) {
  using namespace cdx;
  clear_error();
  const char* name = "cdx_vt_pack";
  if (slabs < 0 || S < 0 || rows < S || S > INT32_MAX - 64)
    return fail(CDX_EINVAL, "%s: bad shape slabs=%lld rows=%lld S=%lld", name, (long long)slabs, (long long)rows,
                (long long)S);
  if (hd <= 0 || hd > 128 || hd % 8 != 0)
    return fail(CDX_EUNSUPPORTED, "%s: head dim %d must be a multiple of 8 and <= 128", name, hd);
  if (vt_ld < S || vt_ld % 64 != 0)
    return fail(CDX_EINVAL, "%s: vt_ld=%lld must be a multiple of 64 that is >= S", name, (long long)vt_ld);
  if (slabs == 0 || S == 0) return CDX_OK;
  const int64_t tiles = (S + 63) / 64;
  if (slabs > INT32_MAX / tiles) return fail(CDX_EUNSUPPORTED, "%s: too many slabs (%lld)", name, (long long)slabs);
  if (!v || !vt) return fail(CDX_EINVAL, "%s: null pointer", name);
  if (!aligned16(v) || !aligned16(vt)) return fail(CDX_EUNSUPPORTED, "%s: pointers must be 16-byte aligned", name);
  vt_pack_kernel<<<dim3((unsigned)(slabs * tiles)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream)>>>(
      v, rows, (int)S, hd, vt, vt_ld);
  return check_launch(name);
}
