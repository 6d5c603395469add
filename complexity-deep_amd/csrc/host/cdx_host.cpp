// Native call paths of the package's operators (module complexity_deep._host).
//
// A forward of few tokens is paced by its host side: checks, output tensors and ctypes
// conversions in Python took 6 to 20 us per operator against 2 to 10 us of kernel time.
// Measured (us per call, issued back to back): 1B attention step of 4 rows 46 -> 22, MoE step
// 32 -> 21, 150M block of 2048 tokens 148 -> 90, 150M model step 1360 -> 762 (with block_step
// 510).
// Each function here is the usual case of one Python operator of the same name: it checks
// its operands, allocates the outputs through torch's allocator, and calls the C-ABI on the
// current stream.  For anything else (a tensor to be made contiguous, cast or broadcast, a
// wrong shape, another device than the current one, an empty call) it launches nothing and
// returns None, and the Python operator goes its general way, which converts or raises.
// Nothing is kept between calls.
#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/utils/pybind.h>

#include <cmath>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../../include/cdx.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

inline void check(int rc, const char* what) {
  if (rc != CDX_OK)
    throw std::runtime_error(std::string(what) + " failed (status " + std::to_string(rc) + "): " + cdx_last_error());
}

// A plain tensor of this dtype on the current device (no wrapper class, storage present).
inline bool plain(const Tensor& t, at::ScalarType dtype = at::kBFloat16) {
  return t.defined() && t.is_cuda() && t.scalar_type() == dtype && t.has_storage() &&
         !t.key_set().has(c10::DispatchKey::Python) && t.get_device() == c10::hip::current_device();
}
inline bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
// Plain, contiguous and 16-byte aligned.
inline bool dense(const Tensor& t, at::ScalarType dtype = at::kBFloat16) {
  return plain(t, dtype) && t.is_contiguous() && aligned(t);
}
inline const uint16_t* u16(const Tensor& t) { return reinterpret_cast<const uint16_t*>(t.data_ptr()); }
inline uint16_t* w16(const Tensor& t) { return reinterpret_cast<uint16_t*>(t.data_ptr()); }
inline const uint16_t* u16(const OptTensor& t) { return t ? u16(*t) : nullptr; }
inline void* stream() { return reinterpret_cast<void*>(c10::hip::getCurrentHIPStream().stream()); }
inline Tensor like(const Tensor& t, at::IntArrayRef shape) { return at::empty(shape, t.options().requires_grad(false)); }
inline Tensor ints(const Tensor& t, at::IntArrayRef shape) {
  return at::empty(shape, t.options().dtype(at::kInt).requires_grad(false));
}

// Row stride of a [..., H] view whose rows are evenly spaced with unit stride inside (0: one
// row for all), or -1.  Dimensions of size 1 have no say: expand() leaves them any stride.
int64_t row_ld(const Tensor& t, int64_t H) {
  if (t.dim() < 1 || t.size(-1) != H || t.stride(-1) != 1) return -1;
  if (t.is_contiguous()) return H;
  int64_t ld = -1, next = 0;
  bool bcast = t.dim() > 1;
  for (int64_t d = t.dim() - 2; d >= 0; --d) {
    if (t.size(d) == 1) continue;
    if (t.stride(d) != 0) bcast = false;
    if (ld < 0)
      ld = t.stride(d);
    else if (t.stride(d) != next)
      return bcast ? 0 : -1;
    next = t.stride(d) * t.size(d);
  }
  if (bcast) return 0;
  if (ld < 0) ld = H;
  return ld < H || ld % 8 != 0 ? -1 : ld;
}

OptTensor rms_norm(const Tensor& x, const Tensor& w, double eps, const OptTensor& out) {
  if (!dense(x) || !dense(w) || x.dim() < 1 || x.numel() == 0) return {};
  const int64_t H = x.size(-1);
  if (w.numel() != H || H % 8 != 0 || H > 8192 || !(eps >= 0)) return {};
  int64_t ldo = H;
  if (out) {
    if (!plain(*out) || !aligned(*out) || out->sizes() != x.sizes()) return {};
    ldo = row_ld(*out, H);
    if (ldo < H) return {};
  }
  Tensor y = out ? *out : like(x, x.sizes());
  check(cdx_rmsnorm_ld_fwd(u16(x), u16(w), (float)eps, x.numel() / H, (int32_t)H, w16(y), ldo, stream()),
        "cdx_rmsnorm_ld_fwd");
  return y;
}

std::optional<std::tuple<Tensor, OptTensor>> add_rms_norm(const Tensor& x, const Tensor& r, const Tensor& w,
                                                          double eps, bool store) {
  if (!dense(x) || !dense(r) || !dense(w) || x.dim() < 1 || x.numel() == 0 || r.sizes() != x.sizes()) return {};
  const int64_t H = x.size(-1);
  if (w.numel() != H || H % 8 != 0 || H > 8192 || !(eps >= 0)) return {};
  Tensor y = like(x, x.sizes());
  OptTensor h;
  if (store) h = like(x, x.sizes());
  check(cdx_add_rmsnorm_fwd(u16(x), u16(r), u16(w), (float)eps, x.numel() / H, (int32_t)H, w16(y),
                            h ? w16(*h) : nullptr, stream()),
        "cdx_add_rmsnorm_fwd");
  return std::make_tuple(y, h);
}

OptTensor embedding(const Tensor& ids, const Tensor& table) {
  if (!plain(ids, at::kLong) || !ids.is_contiguous() || !dense(table) || table.dim() != 2 || ids.numel() == 0) return {};
  const int64_t H = table.size(1);
  if (H % 8 != 0 || H > 16384 || table.size(0) == 0) return {};
  std::vector<int64_t> shape(ids.sizes().begin(), ids.sizes().end());
  shape.push_back(H);
  Tensor out = like(table, shape);
  check(cdx_embedding_fwd(ids.data_ptr<int64_t>(), ids.numel(), u16(table), table.size(0), (int32_t)H, w16(out),
                          stream()),
        "cdx_embedding_fwd");
  return out;
}

OptTensor linear(const Tensor& x, const Tensor& w) {
  if (!dense(x) || !dense(w) || w.dim() != 2 || x.dim() < 2 || x.numel() == 0) return {};
  const int64_t N = w.size(0), K = w.size(1);
  if (x.size(-1) != K || K % 64 != 0 || N % 8 != 0 || N == 0 || N > INT32_MAX || K > INT32_MAX) return {};
  std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = N;
  Tensor out = like(x, shape);
  check(cdx_linear_fwd(u16(x), K, u16(w), K, x.numel() / K, (int32_t)K, (int32_t)N, w16(out), N, stream()),
        "cdx_linear_fwd");
  return out;
}

bool linear_accumulate(const Tensor& x, const Tensor& w, const Tensor& residual) {
  if (!dense(x) || !dense(w) || !dense(residual) || w.dim() != 2 || x.dim() < 2 || x.numel() == 0) return false;
  const int64_t N = w.size(0), K = w.size(1);
  if (x.size(-1) != K || residual.dim() != x.dim() || residual.size(-1) != N ||
      residual.sizes().slice(0, x.dim() - 1) != x.sizes().slice(0, x.dim() - 1) || K % 64 != 0 || N % 8 != 0 || N == 0 ||
      N > INT32_MAX || K > INT32_MAX)
    return false;
  const int64_t M = x.numel() / K;
  if (!cdx_few_rows(M, N)) return false;
  check(cdx_linear_accum_fwd(u16(x), K, u16(w), K, M, (int32_t)K, (int32_t)N, w16(residual), N, stream()),
        "cdx_linear_accum_fwd");
  return true;
}

OptTensor mu_guidance(const Tensor& h, const Tensor& w, const Tensor& mu, double mu_lo, double mu_hi, double lo,
                      double hi, const OptTensor& out) {
  if (!dense(h) || !dense(w) || !dense(mu) || h.dim() < 1 || h.numel() == 0) return {};
  const int64_t H = h.size(-1);
  if (H % 64 != 0 || H > INT32_MAX || mu.dim() != 1 || mu.size(0) != H || w.dim() != 2 || w.size(0) != H ||
      w.size(1) != H || !(lo <= hi) || !(mu_lo <= mu_hi))
    return {};
  int64_t ldo = H;
  if (out) {
    if (!plain(*out) || !aligned(*out) || out->sizes() != h.sizes()) return {};
    ldo = row_ld(*out, H);
    if (ldo < H) return {};
  }
  Tensor y = out ? *out : like(h, h.sizes());
  check(cdx_mu_guidance_fwd(u16(h), h.numel() / H, (int32_t)H, u16(w), u16(mu), (float)mu_lo, (float)mu_hi, (float)lo,
                            (float)hi, w16(y), ldo, stream()),
        "cdx_mu_guidance_fwd");
  return y;
}

using Plan = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>;  // expert_id, perm, inv_perm, counts, offsets

// The plan of ids through a map (without one, ids are expert ids already).
std::optional<Plan> route_plan(const Tensor& ids, const OptTensor& map, int64_t E) {
  const int64_t T = ids.numel();
  if (T == 0 || T > INT32_MAX || E <= 0 || E > 64 || !plain(ids, at::kLong) || !ids.is_contiguous()) return {};
  if (map && (!plain(*map, at::kLong) || !map->is_contiguous() || map->dim() != 1 || map->size(0) == 0)) return {};
  Tensor eid = ints(ids, {T}), perm = ints(ids, {T}), inv = ints(ids, {T}), counts = ints(ids, {E});
  Tensor offsets = ints(ids, {E + 1});
  const size_t bytes = cdx_route_workspace_bytes(T, (int32_t)E);
  Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 16)}, ids.options().dtype(at::kByte));
  check(cdx_route_plan(ids.data_ptr<int64_t>(), T, map ? map->data_ptr<int64_t>() : nullptr, map ? map->size(0) : 0,
                       (int32_t)E, eid.data_ptr<int32_t>(), perm.data_ptr<int32_t>(), inv.data_ptr<int32_t>(),
                       counts.data_ptr<int32_t>(), offsets.data_ptr<int32_t>(), ws.data_ptr(), bytes, stream()),
        "cdx_route_plan");
  return Plan(eid, perm, inv, counts, offsets);
}

// One plan per map over the same ids, each the rows of common buffers.
std::optional<std::vector<Plan>> route_plans(const Tensor& ids, const std::vector<Tensor>& maps, int64_t E) {
  const int64_t L = (int64_t)maps.size(), T = ids.numel();
  if (L == 0 || T == 0 || E <= 0 || E > 64 || L * T > INT32_MAX || !plain(ids, at::kLong) || !ids.is_contiguous())
    return {};
  std::vector<const int64_t*> table;
  table.reserve(L);
  for (const Tensor& m : maps) {
    if (!plain(m, at::kLong) || !m.is_contiguous() || m.dim() != 1 || m.size(0) != maps[0].size(0) || m.size(0) == 0)
      return {};
    table.push_back(m.data_ptr<int64_t>());
  }
  Tensor eid = ints(ids, {L, T}), perm = ints(ids, {L, T}), inv = ints(ids, {L, T});
  Tensor counts = ints(ids, {L, E}), offsets = ints(ids, {L, E + 1});
  const size_t bytes = cdx_route_plans_workspace_bytes(T, (int32_t)E, (int32_t)L);
  Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 16)}, ids.options().dtype(at::kByte));
  check(cdx_route_plans(ids.data_ptr<int64_t>(), T, table.data(), (int32_t)L, maps[0].size(0), (int32_t)E,
                        eid.data_ptr<int32_t>(), perm.data_ptr<int32_t>(), inv.data_ptr<int32_t>(),
                        counts.data_ptr<int32_t>(), offsets.data_ptr<int32_t>(), ws.data_ptr(), bytes, stream()),
        "cdx_route_plans");
  std::vector<Plan> plans;
  plans.reserve(L);
  for (int64_t y = 0; y < L; ++y)
    plans.emplace_back(eid.select(0, y), perm.select(0, y), inv.select(0, y), counts.select(0, y), offsets.select(0, y));
  return plans;
}

OptTensor moe_swiglu(const Tensor& x, const Tensor& perm, const Tensor& offsets, int64_t E, const Tensor& w_gu,
                     const Tensor& w_down, int64_t ie, bool shared, const OptTensor& residual) {
  if (!dense(x) || !dense(w_gu) || !dense(w_down) || x.dim() != 2 || x.numel() == 0 || w_gu.dim() != 4 ||
      w_down.dim() != 3 || !plain(perm, at::kInt) || !plain(offsets, at::kInt) || !perm.is_contiguous() ||
      !offsets.is_contiguous())
    return {};
  const int64_t T = x.size(0), H = x.size(1), P = (ie + 63) / 64 * 64, nb = E + (shared ? 1 : 0);
  if (E <= 0 || E > 64 || H % 64 != 0 || perm.numel() < T || offsets.numel() < E + 1 || w_gu.size(0) != nb ||
      w_gu.size(1) != 2 || w_gu.size(2) != P || w_gu.size(3) != H || w_down.size(0) != nb || w_down.size(1) != H ||
      w_down.size(2) != P)
    return {};
  if (residual && (!dense(*residual) || residual->sizes() != x.sizes())) return {};
  Tensor out = residual ? *residual : like(x, x.sizes());
  Tensor inter = like(x, {T, (shared ? 2 : 1) * P});
  auto fn = residual ? cdx_moe_swiglu_residual_fwd : cdx_moe_swiglu_fwd;
  check(fn(u16(x), T, (int32_t)H, (int32_t)ie, (int32_t)E, shared, perm.data_ptr<int32_t>(),
           offsets.data_ptr<int32_t>(), u16(w_gu), u16(w_down), w16(inter), w16(out), stream()),
        residual ? "cdx_moe_swiglu_residual_fwd" : "cdx_moe_swiglu_fwd");
  return out;
}

// sort_tokens_by_expert: (rows in expert order, their indices, offsets, counts), indices in 64 bits.
std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> sort_tokens(const Tensor& tokens, const Tensor& experts,
                                                                       int64_t E) {
  const int64_t T = experts.numel();
  if (!tokens.is_cuda() || !plain(tokens, tokens.scalar_type()) || !tokens.is_contiguous() || !aligned(tokens) ||
      tokens.dim() < 1 || tokens.size(0) != T || tokens.numel() == 0)
    return {};
  auto plan = route_plan(experts, {}, E);
  if (!plan) return {};
  const auto& [eid, perm, inv, counts, offsets] = *plan;
  Tensor rows = like(tokens, tokens.sizes());
  check(cdx_permute_rows(tokens.data_ptr(), perm.data_ptr<int32_t>(), T, tokens.nbytes() / T, rows.data_ptr(), stream()),
        "cdx_permute_rows");
  auto longs = [&](int64_t n) { return at::empty({n}, experts.options()); };
  Tensor index = longs(T), off64 = longs(E + 1), cnt64 = longs(E);
  check(cdx_widen_plan(perm.data_ptr<int32_t>(), T, offsets.data_ptr<int32_t>(), counts.data_ptr<int32_t>(), (int32_t)E,
                       index.data_ptr<int64_t>(), off64.data_ptr<int64_t>(), cnt64.data_ptr<int64_t>(), stream()),
        "cdx_widen_plan");
  return std::make_tuple(rows, index, off64, cnt64);
}

// persistent_swiglu_cggr: pack the weights and prepare the rows in one launch, then both passes.
OptTensor swiglu_cggr(const Tensor& x, const Tensor& gate, const Tensor& up, const Tensor& down,
                      const Tensor& offsets) {
  if (!dense(x) || x.dim() != 2 || x.numel() == 0 || !dense(gate) || !dense(up) || !dense(down) || gate.dim() != 3 ||
      !plain(offsets, at::kLong) || !offsets.is_contiguous() || offsets.dim() != 1)
    return {};
  const int64_t T = x.size(0), H = x.size(1), E = gate.size(0), I = gate.size(2), P = (I + 63) / 64 * 64;
  if (gate.size(1) != H || up.sizes() != gate.sizes() || down.dim() != 3 || down.size(0) != E || down.size(1) != I ||
      down.size(2) != H || H % 64 != 0 || I % 8 != 0 || I == 0 || E > 64 || E == 0 || offsets.numel() != E + 1 ||
      T > INT32_MAX - 256 || T * H * 2 > (int64_t)UINT32_MAX || E * 2 * P * H * 2 > (int64_t)UINT32_MAX)
    return {};
  Tensor w_gu = like(x, {E, 2, P, H}), w_down = like(x, {E, H, P}), out = like(x, {T, H}), inter = like(x, {T, P});
  Tensor off32 = ints(x, {E + 1}), ident = ints(x, {T});
  void* st = stream();
  check(cdx_cggr_prepare(u16(gate), u16(up), u16(down), (int32_t)E, (int32_t)H, (int32_t)I, offsets.data_ptr<int64_t>(),
                         T, w16(w_gu), w16(w_down), off32.data_ptr<int32_t>(), ident.data_ptr<int32_t>(), w16(out), st),
        "cdx_cggr_prepare");
  check(cdx_moe_swiglu_fwd(u16(x), T, (int32_t)H, (int32_t)I, (int32_t)E, 0, ident.data_ptr<int32_t>(),
                           off32.data_ptr<int32_t>(), u16(w_gu), u16(w_down), w16(inter), w16(out), st),
        "cdx_moe_swiglu_fwd");
  return out;
}

// The attention of a call without a mask, up to o_proj: (merged heads [B, S, nq D], k, v),
// k and v only with a cache.  w is the [N, 2 H] buffer of the projection and mu weights side
// by side.  past: both or neither.  Covers the fused projection (heads of 32, 64 and 128)
// and the few-row / other-head-dim form, chosen as in ComplexityAttention.forward.
std::optional<std::tuple<Tensor, OptTensor, OptTensor>> attention(
    const Tensor& x, const OptTensor& mu_in, const Tensor& w, int64_t nq, int64_t nkv, int64_t D, const OptTensor& qn,
    const OptTensor& kn, double eps, const Tensor& cos_sin, const OptTensor& past_k, const OptTensor& past_v,
    bool use_cache) {
  if (!plain(x) || !aligned(x) || x.dim() != 3 || x.numel() == 0 || !dense(w) || w.dim() != 2) return {};
  const int64_t B = x.size(0), S = x.size(1), H = x.size(2), M = B * S, N = (nq + 2 * nkv) * D;
  if (H % 64 != 0 || w.size(0) != N || w.size(1) != 2 * H || nkv <= 0 || nq % nkv != 0 || D <= 0 || D % 8 != 0 ||
      D > 128)
    return {};
  const int64_t ldx = row_ld(x, H);
  if (ldx < H) return {};
  OptTensor mu = mu_in;
  int64_t ldmu = 0;
  if (mu) {
    if (!plain(*mu) || !aligned(*mu) || mu->dim() != 3 || mu->size(0) != B || mu->size(1) != S || mu->size(2) != H)
      return {};
    ldmu = row_ld(*mu, H);
    if (ldmu < 0) return {};
    if (ldmu == 0 && M == 1) ldmu = H;
  }
  if (qn.has_value() != kn.has_value()) return {};
  if (qn && (!dense(*qn) || !dense(*kn) || qn->numel() != D || kn->numel() != D)) return {};
  if (past_k.has_value() != past_v.has_value() || (past_k && past_k->dim() != 4)) return {};
  const int64_t P = past_k ? past_k->size(2) : 0;
  if (!plain(cos_sin, at::kFloat) || !cos_sin.is_contiguous() || cos_sin.size(0) < P + S || !(eps >= 0)) return {};
  const float scale = (float)(1.0 / std::sqrt((double)D));
  const uint16_t* w_mu = u16(w) + H;
  const int64_t ldw = 2 * H, vt_ld = (S + 63) / 64 * 64, n_pos = cos_sin.size(0);
  const float* table = cos_sin.data_ptr<float>();
  void* st = stream();
  const bool fused_dim = D == 32 || D == 64 || D == 128, few = cdx_few_rows(M, N) != 0;

  if (fused_dim && !few && !past_k && !use_cache) {
    Tensor q = like(x, {B, nq, S, D}), k = like(x, {B, nkv, S, D}), vt = like(x, {B, nkv, D, vt_ld});
    // Columns of the key positions S .. vt_ld - 1 are masked but must be finite (the order
    // inside a 16-group moves some of them below S).
    if (vt_ld > S) vt.narrow(3, S / 16 * 16, vt_ld - S / 16 * 16).zero_();
    const bool side = mu && ldmu == ldx && ldx >= 2 * H && mu->data_ptr() == static_cast<const void*>(u16(x) + H);
    if (mu && ldmu == 0 && H > 64) {
      Tensor work = like(x, {N * ldw + 64});
      check(cdx_mu_qkv_rope_bcast_fwd(u16(x), ldx, u16(*mu), u16(w), w_mu, ldw, B, S, (int32_t)H, (int32_t)nq,
                                      (int32_t)nkv, (int32_t)D, u16(qn), u16(kn), (float)eps, table, n_pos, 0, w16(q),
                                      w16(k), w16(vt), vt_ld, w16(work), st),
            "cdx_mu_qkv_rope_bcast_fwd");
    } else {
      check(cdx_mu_qkv_rope_fwd(u16(x), ldx, side ? nullptr : u16(mu), side ? 0 : ldmu, u16(w), side ? nullptr : w_mu,
                                ldw, B, S, (int32_t)(side ? 2 * H : H), (int32_t)nq, (int32_t)nkv, (int32_t)D, u16(qn),
                                u16(kn), (float)eps, table, n_pos, 0, w16(q), w16(k), w16(vt), vt_ld, st),
            "cdx_mu_qkv_rope_fwd");
    }
    Tensor out = like(x, {B, S, nq * D});
    check(cdx_attention_fwd(u16(q), u16(k), u16(vt), B, S, (int32_t)nq, (int32_t)nkv, (int32_t)D, vt_ld, scale,
                            w16(out), st),
          "cdx_attention_fwd");
    return std::make_tuple(out, OptTensor(), OptTensor());
  }
  if (fused_dim && !few) return {};  // a long prompt into a cache
  if (past_k && (!dense(*past_k) || !dense(*past_v) || past_k->dim() != 4 || past_k->size(0) != B ||
                 past_k->size(1) != nkv || past_k->size(3) != D || past_v->sizes() != past_k->sizes() || P == 0 ||
                 (at::GradMode::is_enabled() && (past_k->requires_grad() || past_v->requires_grad()))))
    return {};
  if (2 * B * nkv * (P + S) > INT32_MAX / (D / 8) || M > INT32_MAX / (nq + 2 * nkv)) return {};
  const bool attend = S <= 16 && P >= S;
  OptTensor q;
  if (!attend) q = like(x, {B, nq, S, D});
  Tensor out = like(x, {B, S, nq * D});
  Tensor k = like(x, {B, nkv, P + S, D}), v = like(x, {B, nkv, P + S, D});
  const size_t bytes = cdx_qkv_cache_workspace_bytes(B, S, (int32_t)nq, (int32_t)nkv, (int32_t)D);
  Tensor work = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte).requires_grad(false));
  Tensor vt;
  if (!attend) vt = like(x, {B, nkv, D, vt_ld});
  if (!attend && P == 0) {
    check(cdx_qkv_prompt_fwd(u16(x), ldx, u16(mu), ldmu, u16(w), w_mu, ldw, B, S, (int32_t)H, (int32_t)nq, (int32_t)nkv,
                             (int32_t)D, u16(qn), u16(kn), (float)eps, table, n_pos, w16(*q), w16(k), w16(v), w16(vt),
                             vt_ld, work.data_ptr(), bytes, st),
          "cdx_qkv_prompt_fwd");
  } else {
    check(cdx_qkv_cache_fwd(u16(x), ldx, u16(mu), ldmu, u16(w), w_mu, ldw, B, S, (int32_t)H, (int32_t)nq, (int32_t)nkv,
                            (int32_t)D, u16(qn), u16(kn), (float)eps, table, n_pos, u16(past_k), u16(past_v), P,
                            q ? w16(*q) : nullptr, w16(k), w16(v), attend ? w16(out) : nullptr, scale, work.data_ptr(),
                            bytes, st),
          "cdx_qkv_cache_fwd");
    if (!attend) check(cdx_vt_pack(u16(v), B * nkv, P + S, S, (int32_t)D, w16(vt), vt_ld, st), "cdx_vt_pack");
  }
  if (!attend)
    check(cdx_attention_cache_fwd(u16(*q), u16(k), u16(vt), B, S, P + S, (int32_t)nq, (int32_t)nkv, (int32_t)D, vt_ld,
                                  scale, w16(out), st),
          "cdx_attention_cache_fwd");
  return std::make_tuple(out, OptTensor(k), OptTensor(v));
}

// One decoder block of a generation step (B * S <= 8), h updated in place: the input norm, the
// attention with its cache, o_proj and its residual add, the post-attention norm, the MoE and
// its residual add, and mu for the next layer (with mu_w), in six launches: both norms are
// folded into the products that read them.  Returns (k, v, mu).
std::optional<std::tuple<Tensor, Tensor, OptTensor>> block_step(
    const Tensor& h, const Tensor& ln1, double eps1, const OptTensor& mu, const Tensor& w, int64_t nq, int64_t nkv,
    int64_t D, const OptTensor& qn, const OptTensor& kn, double qk_eps, const Tensor& cos_sin,
    const OptTensor& past_k, const OptTensor& past_v, const Tensor& o_w, const Tensor& ln2, double eps2,
    const Tensor& perm, const Tensor& offsets, int64_t E, const Tensor& w_gu, const Tensor& w_down, int64_t ie,
    bool shared, const OptTensor& mu_w, const OptTensor& mu_param, double mu_lo, double mu_hi, double lo, double hi) {
  if (!dense(h) || h.dim() != 3 || h.numel() == 0 || !dense(ln1) || !dense(ln2) || !dense(w) || !dense(o_w) ||
      !dense(w_gu) || !dense(w_down) || w.dim() != 2 || o_w.dim() != 2 || w_gu.dim() != 4 || w_down.dim() != 3)
    return {};
  const int64_t B = h.size(0), S = h.size(1), H = h.size(2), M = B * S, N = (nq + 2 * nkv) * D;
  if (M > 8 || !cdx_few_rows(M, N) || !cdx_few_rows(M, H) || H % 64 != 0 || H > 8192 || ln1.numel() != H ||
      ln2.numel() != H || nkv <= 0 || nq % nkv != 0 || D <= 0 || D % 8 != 0 || D > 128 || w.size(0) != N ||
      w.size(1) != 2 * H || o_w.size(0) != H || o_w.size(1) != nq * D || (nq * D) % 64 != 0 || !(eps1 >= 0) ||
      !(eps2 >= 0) || !(qk_eps >= 0))
    return {};
  int64_t ldmu = 0;
  if (mu) {
    if (!plain(*mu) || !aligned(*mu) || mu->dim() != 3 || mu->size(0) != B || mu->size(1) != S || mu->size(2) != H)
      return {};
    ldmu = row_ld(*mu, H);
    if (ldmu < 0) return {};
  }
  if (qn.has_value() != kn.has_value() || past_k.has_value() != past_v.has_value()) return {};
  if (qn && (!dense(*qn) || !dense(*kn) || qn->numel() != D || kn->numel() != D)) return {};
  if (past_k && (!dense(*past_k) || !dense(*past_v) || past_k->dim() != 4 || past_k->size(0) != B ||
                 past_k->size(1) != nkv || past_k->size(2) == 0 || past_k->size(3) != D ||
                 past_v->sizes() != past_k->sizes() ||
                 (at::GradMode::is_enabled() && (past_k->requires_grad() || past_v->requires_grad()))))
    return {};
  const int64_t past = past_k ? past_k->size(2) : 0;
  if (!plain(cos_sin, at::kFloat) || !cos_sin.is_contiguous() || cos_sin.size(0) < past + S ||
      2 * B * nkv * (past + S) > INT32_MAX / (D / 8))
    return {};
  const int64_t P = (ie + 63) / 64 * 64, nb = E + (shared ? 1 : 0);
  if (!plain(perm, at::kInt) || !plain(offsets, at::kInt) || !perm.is_contiguous() || !offsets.is_contiguous() ||
      perm.numel() < M || E <= 0 || E > 64 || offsets.numel() < E + 1 || w_gu.size(0) != nb || w_gu.size(1) != 2 ||
      w_gu.size(2) != P || w_gu.size(3) != H || w_down.size(0) != nb || w_down.size(1) != H || w_down.size(2) != P)
    return {};
  if (mu_w && (!mu_param || !dense(*mu_w) || !dense(*mu_param) || mu_w->dim() != 2 || mu_w->size(0) != H ||
               mu_w->size(1) != H || mu_param->dim() != 1 || mu_param->size(0) != H || !(lo <= hi) || !(mu_lo <= mu_hi)))
    return {};

  void* st = stream();
  const float scale = (float)(1.0 / std::sqrt((double)D));
  const bool attend = S <= 16 && past >= S;
  Tensor attn = like(h, {B, S, nq * D}), k = like(h, {B, nkv, past + S, D}), v = like(h, {B, nkv, past + S, D});
  OptTensor q;
  if (!attend) q = like(h, {B, nq, S, D});
  const size_t bytes = cdx_qkv_cache_workspace_bytes(B, S, (int32_t)nq, (int32_t)nkv, (int32_t)D);
  Tensor work = at::empty({(int64_t)bytes}, h.options().dtype(at::kByte).requires_grad(false));
  check(cdx_qkv_cache_norm_fwd(u16(h), H, u16(ln1), (float)eps1, u16(mu), ldmu, u16(w), u16(w) + H, 2 * H, B, S,
                               (int32_t)H, (int32_t)nq, (int32_t)nkv, (int32_t)D, u16(qn), u16(kn), (float)qk_eps,
                               cos_sin.data_ptr<float>(), cos_sin.size(0), u16(past_k), u16(past_v), past,
                               q ? w16(*q) : nullptr, w16(k), w16(v), attend ? w16(attn) : nullptr, scale,
                               work.data_ptr(), bytes, st),
        "cdx_qkv_cache_norm_fwd");
  if (!attend) {
    Tensor vt = like(h, {B, nkv, D, 64});  // S <= 8
    check(cdx_vt_pack(u16(v), B * nkv, past + S, S, (int32_t)D, w16(vt), 64, st), "cdx_vt_pack");
    check(cdx_attention_cache_fwd(u16(*q), u16(k), u16(vt), B, S, past + S, (int32_t)nq, (int32_t)nkv, (int32_t)D, 64,
                                  scale, w16(attn), st),
          "cdx_attention_cache_fwd");
  }
  check(cdx_linear_accum_fwd(u16(attn), nq * D, u16(o_w), nq * D, M, (int32_t)(nq * D), (int32_t)H, w16(h), H, st),
        "cdx_linear_accum_fwd");
  Tensor inter = like(h, {M, (shared ? 2 : 1) * P});
  check(cdx_moe_swiglu_norm_residual_fwd(w16(h), u16(ln2), (float)eps2, M, (int32_t)H, (int32_t)ie, (int32_t)E, shared,
                                         perm.data_ptr<int32_t>(), offsets.data_ptr<int32_t>(), u16(w_gu),
                                         u16(w_down), w16(inter), st),
        "cdx_moe_swiglu_norm_residual_fwd");
  OptTensor mu_out;
  if (mu_w) {
    mu_out = like(h, h.sizes());
    check(cdx_mu_guidance_fwd(u16(h), M, (int32_t)H, u16(*mu_w), u16(*mu_param), (float)mu_lo, (float)mu_hi, (float)lo,
                              (float)hi, w16(*mu_out), H, st),
          "cdx_mu_guidance_fwd");
  }
  return std::make_tuple(k, v, mu_out);
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("rms_norm", &rms_norm);
  m.def("add_rms_norm", &add_rms_norm);
  m.def("embedding", &embedding);
  m.def("linear", &linear);
  m.def("linear_accumulate", &linear_accumulate);
  m.def("mu_guidance", &mu_guidance);
  m.def("route_plan", &route_plan);
  m.def("route_plans", &route_plans);
  m.def("moe_swiglu", &moe_swiglu);
  m.def("sort_tokens", &sort_tokens);
  m.def("swiglu_cggr", &swiglu_cggr);
  m.def("attention", &attention);
  m.def("block_step", &block_step);
}
