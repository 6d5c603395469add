// Expert weights laid out [experts][in][out] (the operator API's) moved into the layouts the
// MoE kernels read (gfx950): w_gu [E][2][P][H] and w_down [E][H][P], units in [I, P) zero.
//
// Reference behaviour: cuda/persistent_cggr.py:479-530 takes the weights as arguments of each
// call, so the move is part of every call.  All three operands go in one launch of 64 x 64
// transposes: 16-byte reads along the source rows, the tile in LDS, 16-byte writes along the
// destination rows.  The same launch prepares what else persistent_swiglu_cggr needs: the
// segment offsets in 32 bits, an identity permutation and zeros in the output rows that no
// segment covers (three launches and 9 us before; sort + experts at 4096 tokens 63 -> 46.5 us
// with the plan's indices widened by one launch too).  Bound: one read and one write of the
// weights.  Measured for 4 experts of 768 x 512 (9.4 MB each way): 8.0 us, with the rows'
// preparation 9.6; three strided tensor copies and two clears took 42 us.
#include "cdx_common.h"

namespace cdx {
namespace {

constexpr int kTile = 64;
constexpr int kPitch = kTile + 8;  // LDS row of 144 bytes: 16-byte aligned, rows on shifted banks

struct PackParams {
  const uint16_t* gate;  // [E][H][I]
  const uint16_t* up;    // [E][H][I]
  const uint16_t* down;  // [E][I][H]
  uint16_t* w_gu;
  uint16_t* w_down;
  int32_t H, I, P;
  // With out: E + 1 segment offsets, the identity permutation of T rows, and the output.
  const int64_t* offsets;
  int32_t* offsets32;
  int32_t* ident;
  uint16_t* out;
  int32_t E, T;
};

__device__ __forceinline__ int row_index(int64_t v, int T) { return (int)(v < 0 ? 0 : (v > T ? T : v)); }

// Rows [256 b, 256 b + 256) of the identity and of the output; block 0 the offsets too.
__device__ void prepare_rows(const PackParams& p, int b) {
  if (b == 0)
    for (int x = threadIdx.x; x <= p.E; x += 256) p.offsets32[x] = row_index(p.offsets[x], p.T);
  const int row = b * 256 + threadIdx.x;
  if (row < p.T) p.ident[row] = row;
  const int lo = row_index(p.offsets[0], p.T), hi = row_index(p.offsets[p.E], p.T);
  const int r0 = b * 256, r1 = min(p.T, r0 + 256);
  if (lo <= r0 && r1 <= hi) return;
  const int vecs = p.H / 8;
  for (int i = threadIdx.x; i < (r1 - r0) * vecs; i += 256) {
    const int r = r0 + i / vecs;
    if (r < lo || r >= hi)
      reinterpret_cast<uint4*>(p.out + (int64_t)r * p.H)[i % vecs] = make_uint4(0u, 0u, 0u, 0u);
  }
}

// Block (tile, operand, expert): destination rows [r0, r0 + 64) x columns [c0, c0 + 64) of a
// matrix whose element (r, c) is source element (c, r), zero outside the source.
__global__ __launch_bounds__(256) void moe_pack_kernel(const PackParams p) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[kTile * kPitch];
  const int e = blockIdx.z, which = blockIdx.y;
  if (which == 3) {
    // The (tile, expert) blocks of this plane share the rows.
    const int step = gridDim.x * gridDim.z;
    for (int b = blockIdx.z * gridDim.x + blockIdx.x; b * 256 < p.T || b == 0; b += step) prepare_rows(p, b);
    return;
  }
  const int64_t src_size = (int64_t)p.H * p.I, dst_size = (int64_t)p.H * p.P;
  const uint16_t* src = (which == 0 ? p.gate : (which == 1 ? p.up : p.down)) + e * src_size;
  uint16_t* dst = which == 2 ? p.w_down + e * dst_size : p.w_gu + (2 * (int64_t)e + which) * dst_size;
  const int src_cols = which == 2 ? p.H : p.I;  // source row length
  const int src_rows = which == 2 ? p.I : p.H;
  const int dst_cols = which == 2 ? p.P : p.H;
  const int tiles_c = dst_cols / kTile;
  const int r0 = (int)(blockIdx.x / tiles_c) * kTile, c0 = (int)(blockIdx.x % tiles_c) * kTile;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int t = threadIdx.x + i * 256, row = t >> 3, ch = t & 7;
    // Source row c0 + row, columns r0 + 8 ch .. + 7 (both counts are multiples of 8).
    const bool in = c0 + row < src_rows && r0 + ch * 8 < src_cols;
    const uint4 v = *reinterpret_cast<const uint4*>(src + (in ? (int64_t)(c0 + row) * src_cols + r0 + ch * 8 : 0));
    *reinterpret_cast<uint4*>(tile + row * kPitch + ch * 8) = in ? v : make_uint4(0u, 0u, 0u, 0u);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int t = threadIdx.x + i * 256, row = t >> 3, ch = t & 7;
    const uint16_t* q = tile + ch * 8 * kPitch + row;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = (uint32_t)q[2 * j * kPitch] | ((uint32_t)q[(2 * j + 1) * kPitch] << 16);
    *reinterpret_cast<uint4*>(dst + (int64_t)(r0 + row) * dst_cols + c0 + ch * 8) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

}  // namespace
}  // namespace cdx

namespace cdx {
namespace {

int moe_pack(const char* name, const uint16_t* gate, const uint16_t* up, const uint16_t* down, int32_t E, int32_t H,
             int32_t I, uint16_t* w_gu, uint16_t* w_down, const int64_t* offsets, int64_t T, int32_t* offsets32,
             int32_t* ident, uint16_t* out, void* stream) {
  if (E <= 0 || H <= 0 || I <= 0) return fail(CDX_EINVAL, "%s: bad shape E=%d H=%d I=%d", name, E, H, I);
  if (H % kTile != 0 || I % 8 != 0 || E > 65535 || I > INT32_MAX - 64)
    return fail(CDX_EUNSUPPORTED, "%s: H=%d must be a multiple of 64 and I=%d of 8", name, H, I);
  if (!gate || !up || !down || !w_gu || !w_down) return fail(CDX_EINVAL, "%s: null pointer", name);
  if (!aligned16(gate) || !aligned16(up) || !aligned16(down) || !aligned16(w_gu) || !aligned16(w_down))
    return fail(CDX_EUNSUPPORTED, "%s: pointers must be 16-byte aligned", name);
  PackParams p{gate, up, down, w_gu, w_down, H, I, (I + 63) / 64 * 64, offsets, offsets32, ident, out, E, (int32_t)T};
  const int64_t tiles = (int64_t)(H / kTile) * (p.P / kTile);
  if (tiles > INT32_MAX) return fail(CDX_EUNSUPPORTED, "%s: problem too large", name);
  moe_pack_kernel<<<dim3((unsigned)tiles, out ? 4 : 3, (unsigned)E), dim3(256), 0,
                    reinterpret_cast<hipStream_t>(stream)>>>(p);
  return check_launch(name);
}

}  // namespace
}  // namespace cdx

extern "C" int cdx_moe_pack(const uint16_t* gate, const uint16_t* up, const uint16_t* down, int32_t E, int32_t H,
                            int32_t I, uint16_t* w_gu, uint16_t* w_down, void* stream) {
  cdx::clear_error();
  return cdx::moe_pack("cdx_moe_pack", gate, up, down, E, H, I, w_gu, w_down, nullptr, 0, nullptr, nullptr, nullptr,
                       stream);
}

extern "C" int cdx_cggr_prepare(const uint16_t* gate, const uint16_t* up, const uint16_t* down, int32_t E, int32_t H,
                                int32_t I, const int64_t* offsets, int64_t T, uint16_t* w_gu, uint16_t* w_down,
                                int32_t* offsets32, int32_t* ident, uint16_t* out, void* stream) {
  using namespace cdx;
  clear_error();
  const char* name = "cdx_cggr_prepare";
  if (T <= 0 || T > INT32_MAX - 256) return fail(CDX_EINVAL, "%s: T=%lld out of range", name, (long long)T);
  if (!offsets || !offsets32 || !ident || !out) return fail(CDX_EINVAL, "%s: null pointer", name);
  if (!aligned16(out)) return fail(CDX_EUNSUPPORTED, "%s: pointers must be 16-byte aligned", name);
  return moe_pack(name, gate, up, down, E, H, I, w_gu, w_down, offsets, T, offsets32, ident, out, stream);
}
