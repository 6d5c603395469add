"""GQA attention with the mu-guided QKV projection on the gfx950 kernel (piece 2).

Interfaces follow the reference:
  ComplexityAttention        core/attention.py:33-181 (constructor, parameters and
                             state_dict keys; exported also as MuGuidedAttention)
  fused_mu_qkv_projection    cuda/triton_mu_qkv.py:195-283 (weights [in, out])
  FusedMuQKVProjection       cuda/triton_mu_qkv.py:336-394

The projection is one MFMA contraction over K = 2H: [x | mu_prev] @ [W_x | W_mu]^T
with W_x = [Wq; Wk; Wv] and W_mu = [Wmu_q; Wmu_k; Wmu_v], the kernel switching weight
source at K = H.  The module keeps W_x and W_mu side by side in one [N, 2H] buffer
(row n is [W_x[n] | W_mu[n]], the layout of the reference's torch.cat(..., dim=1)) and
its six Linear weights are views of it, so nothing is concatenated per forward
(attention.py:122-124 concatenates every call) and every write to a weight, through
``.data`` or otherwise, reaches the kernel operand.  When x and mu also sit side by
side in one [T, 2H] buffer (the model writes them so), the projection is one plain
K = 2H contraction over single operands.  q, k and v are column slices of
the packed [T, Nq*D + 2*Nkv*D] output.

ComplexityAttention.forward goes one step further for head dims 32/64/128: the
per-head QK RMSNorm and RoPE (attention.py:138-155) run in the projection kernel's
epilogue (cdx_mu_qkv_rope_fwd), which writes q, k, v head-major, in fp32 up to one
final rounding.  The few rows of a generation step, and heads of other dims (multiples of
8 up to 128), go through cdx_qkv_cache_fwd: the product, then one pass that normalises,
rotates and extends the KV cache.  Without a mask the attention is the causal kernel's,
with or without a cache: its mask is aligned at the top left, as is_causal=True aligns it
for more keys than queries (attention.py:168-175), so query i sees keys 0 .. i of the
cache.  Attention with a mask stays PyTorch-ROCm's SDPA (attention.py:157-181), and o_proj
of more than a few rows a library GEMM.
"""

from __future__ import annotations

import sys
from typing import Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _native as nat
from ._grad import forward_only
from .linear import few_rows, linear, linear_accumulate_
from .rotary import RotaryEmbedding, apply_rotary_pos_emb


def _rows_view(t: torch.Tensor, H: int) -> Tuple[torch.Tensor, int]:
    """Express a [..., H] tensor as rows base + r * ld; ld = 0 for one broadcast row.
    (Only the base pointer and ld are used: a contiguous tensor is returned as is.)"""
    if t.shape[-1] == H and t.is_contiguous():
        return t, H
    if t.stride(-1) != 1:
        return t.contiguous(), H
    # (Dimensions of size 1 have no say: expand() leaves them any stride.)
    if t.dim() > 1 and all(s == 0 for n, s in zip(t.shape[:-1], t.stride()[:-1]) if n != 1):
        return t, 0
    try:
        rows = t.view(-1, H)
    except RuntimeError:
        rows = t.contiguous().view(-1, H)
    ld = rows.stride(0) if rows.shape[0] > 1 else H
    if ld < H:
        rows = rows.contiguous()
        ld = H
    return rows, ld


def _weight_sources(w: torch.Tensor, w_mu: Optional[torch.Tensor], mu: Optional[torch.Tensor], H: int,
                    what: str) -> Tuple[int, Optional[int], int]:
    """(x-weight pointer, mu-weight pointer, common row stride) for the kernels.

    ``w`` is [N, >= H] (unit stride in K).  With ``w_mu`` None and a mu operand, ``w``
    is a packed [N, >= 2H] whose columns [H, 2H) are the mu weights; otherwise
    ``w_mu`` is [N, H] with the same row stride as ``w``."""
    if w.dim() != 2 or w.stride(-1) != 1 or w.shape[1] < H:
        raise ValueError(f"{what}: weight must be [N, >= {H}] with unit stride in K")
    ldw = w.stride(0) if w.shape[0] > 1 else w.shape[1]
    if mu is None:
        return w.data_ptr(), None, ldw
    if w_mu is None:
        if w.shape[1] < 2 * H:
            raise ValueError(f"{what}: a packed weight needs 2H = {2 * H} columns, got {w.shape[1]}")
        return w.data_ptr(), w.data_ptr() + H * w.element_size(), ldw
    if w_mu.dim() != 2 or w_mu.shape[0] != w.shape[0] or w_mu.shape[1] < H:
        raise ValueError(f"{what}: mu weight shape {tuple(w_mu.shape)} does not match {tuple(w.shape)}")
    ldm = w_mu.stride(0) if w_mu.shape[0] > 1 else ldw
    if w_mu.stride(-1) != 1 or ldm != ldw or w_mu.dtype != w.dtype or w_mu.device != w.device:
        raise ValueError(f"{what}: x and mu weights must share dtype, device and row stride")
    return w.data_ptr(), w_mu.data_ptr(), ldw


def _check_widths(x: torch.Tensor, mu: Optional[torch.Tensor], H: int, what: str) -> None:
    """The kernels read rows of H values through the base pointers of x and mu."""
    if x.shape[-1] != H:
        raise ValueError(f"{what}: x hidden size {x.shape[-1]} != {H}")
    if mu is not None and mu.shape[-1] != H:
        raise ValueError(f"{what}: mu hidden size {mu.shape[-1]} != {H}")


def mu_qkv_project(x: torch.Tensor, mu: Optional[torch.Tensor], w_pack: torch.Tensor,
                   H: int, w_mu: Optional[torch.Tensor] = None) -> torch.Tensor:
    """[..., N] = [x | mu] @ [w_x | w_mu]^T (cdx_mu_qkv_fwd).

    w_pack is [N, 2H] (x weights then mu weights) or, with ``w_mu`` given, the x
    weights [N, H] alone; with mu=None only its first H columns are read."""
    nat.require_device(x, mu, w_pack, w_mu, what="mu_qkv_project")
    _check_widths(x, mu, H, "mu_qkv_project")
    lead = x.shape[:-1]
    x2, ldx = _rows_view(x, H)
    if ldx == 0:
        x2, ldx = x.contiguous(), H
    M = x.numel() // H
    N = w_pack.shape[0]
    if mu is not None:
        mu = mu.expand(*lead, H) if mu.shape[:-1] != lead else mu
        mu2, ldmu = _rows_view(mu, H)
    else:
        mu2, ldmu = None, 0
    wx_ptr, wmu_ptr, ldw = _weight_sources(w_pack, w_mu, mu2, H, "mu_qkv_project")
    out = torch.empty(*lead, N, dtype=x.dtype, device=x.device)
    with nat.launch_region("mu_qkv", x.device, M=M, H=H, N=N, mu=mu2 is not None):
        nat.check(nat.lib().cdx_mu_qkv_fwd(x2.data_ptr(), ldx, nat.ptr(mu2), ldmu, wx_ptr, wmu_ptr, ldw,
                                           M, H, N, out.data_ptr(), N, nat.stream_of(x)), "cdx_mu_qkv_fwd")
    return out


def vt_ld_for(S: int) -> int:
    """Row length of the transposed V layout (keys padded to a multiple of 64)."""
    return (S + 63) // 64 * 64


def vt_columns(S: int, device=None) -> torch.Tensor:
    """Column of each token s in the transposed V layout: inside every group of 16 the
    middle two groups of 4 swap places (the key order of the attention kernel's
    P fragments)."""
    s = torch.arange(S, device=device)
    q = (s // 4) % 4
    qs = torch.where(q == 1, 2, torch.where(q == 2, 1, q))
    return (s // 16) * 16 + 4 * qs + s % 4


def to_vt_layout(v: torch.Tensor) -> torch.Tensor:
    """[B, h, S, D] -> the transposed layout [B, h, D, vt_ld] cdx_attention_fwd reads
    (padding columns zero).  The model never calls this: the projection kernel writes
    V in this layout directly."""
    B, h, S, D = v.shape
    vt = torch.zeros(B, h, D, vt_ld_for(S), dtype=v.dtype, device=v.device)
    vt[..., vt_columns(S, v.device)] = v.transpose(-1, -2)
    return vt


def mu_qkv_rope(x: torch.Tensor, mu: Optional[torch.Tensor], w_pack: torch.Tensor, H: int, nq: int,
                nkv: int, hd: int, q_norm_w: Optional[torch.Tensor], k_norm_w: Optional[torch.Tensor],
                eps: float, cos_sin: torch.Tensor, pos0: int = 0, v_transposed: bool = False,
                w_mu: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(q, k, v) head-major [B, heads, S, hd] from x [B, S, H] (cdx_mu_qkv_rope_fwd):
    the mu-QKV projection with per-head RMSNorm of q and k (weights q_norm_w /
    k_norm_w, None = no norm) and RoPE at positions pos0 .. pos0+S-1 fused into one
    kernel.  cos_sin is the fp32 [n_pos, hd/2, 2] table of RotaryEmbedding.  Weights
    as in mu_qkv_project.  v_transposed=True returns V in the layout of to_vt_layout
    instead.  A mu that is one row broadcast to every token (layer 0's mu_init.expand)
    goes through cdx_mu_qkv_rope_bcast_fwd, which folds its product with W_mu into one
    64-column K block (K = H + 64 instead of 2H)."""
    nat.require_device(x, mu, w_pack, w_mu, q_norm_w, k_norm_w, what="mu_qkv_rope")
    _check_widths(x, mu, H, "mu_qkv_rope")
    if w_pack.shape[0] != (nq + 2 * nkv) * hd:
        raise ValueError(f"mu_qkv_rope: weight has {w_pack.shape[0]} rows, {nq} + 2 x {nkv} heads of {hd} need "
                         f"{(nq + 2 * nkv) * hd}")
    B, S, _ = x.shape
    x2, ldx = _rows_view(x, H)
    if ldx == 0:
        x2, ldx = x.contiguous(), H
    if mu is not None:
        mu = mu.expand(B, S, H) if mu.shape[:-1] != (B, S) else mu
        mu2, ldmu = _rows_view(mu, H)
    else:
        mu2, ldmu = None, 0
    wx_ptr, wmu_ptr, ldw = _weight_sources(w_pack, w_mu, mu2, H, "mu_qkv_rope")
    if cos_sin.dtype != torch.float32 or not cos_sin.is_contiguous() or cos_sin.device != x.device:
        raise ValueError("mu_qkv_rope: cos_sin must be a contiguous fp32 table on the input's device")
    if (q_norm_w is None) != (k_norm_w is None):
        raise ValueError("mu_qkv_rope: pass both QK norm weights or neither")
    if q_norm_w is not None:
        q_norm_w = q_norm_w.to(x.dtype).contiguous()
        k_norm_w = k_norm_w.to(x.dtype).contiguous()
    q = torch.empty(B, nq, S, hd, dtype=x.dtype, device=x.device)
    k = torch.empty(B, nkv, S, hd, dtype=x.dtype, device=x.device)
    if v_transposed:
        vt_ld = vt_ld_for(S)
        v = torch.empty(B, nkv, hd, vt_ld, dtype=x.dtype, device=x.device)
        if vt_ld > S:
            # Columns of the key positions S .. vt_ld-1 are masked but must be finite.
            # The order inside a 16-group moves some of them below S, so clear from the
            # last partial group on; the kernel then fills the columns of tokens < S.
            v[..., (S // 16) * 16:].zero_()
    else:
        vt_ld = 0
        v = torch.empty(B, nkv, S, hd, dtype=x.dtype, device=x.device)
    N = (nq + 2 * nkv) * hd
    esz = x.element_size()
    if (mu2 is not None and ldmu != 0 and ldx == ldmu and ldx >= 2 * H and ldw >= 2 * H
            and mu2.data_ptr() == x2.data_ptr() + H * esz and wmu_ptr == wx_ptr + H * esz):
        # x and mu side by side in one buffer, and W_x and W_mu likewise: one K = 2H
        # contraction over single operands (the same sums in the same order).
        with nat.launch_region("mu_qkv", x.device, M=B * S, H=H, N=N, mu=True):
            nat.check(nat.lib().cdx_mu_qkv_rope_fwd(
                x2.data_ptr(), ldx, None, 0, wx_ptr, None, ldw, B, S, 2 * H, nq, nkv, hd,
                nat.ptr(q_norm_w), nat.ptr(k_norm_w), float(eps), cos_sin.data_ptr(), cos_sin.shape[0], pos0,
                q.data_ptr(), k.data_ptr(), v.data_ptr(), vt_ld, nat.stream_of(x)), "cdx_mu_qkv_rope_fwd")
        return q, k, v
    if mu2 is not None and ldmu == 0 and H > 64:
        # One broadcast mu row (layer 0's mu_init.expand): its product with W_mu is one
        # row, folded into a 64-column K block (K = H + 64 instead of 2H).
        work = torch.empty(N * ldw + 64, dtype=x.dtype, device=x.device)
        with nat.launch_region("mu_qkv_bcast", x.device, M=B * S, H=H, N=N):
            nat.check(nat.lib().cdx_mu_qkv_rope_bcast_fwd(
                x2.data_ptr(), ldx, mu2.data_ptr(), wx_ptr, wmu_ptr, ldw, B, S, H, nq, nkv, hd,
                nat.ptr(q_norm_w), nat.ptr(k_norm_w), float(eps), cos_sin.data_ptr(), cos_sin.shape[0], pos0,
                q.data_ptr(), k.data_ptr(), v.data_ptr(), vt_ld, work.data_ptr(), nat.stream_of(x)),
                "cdx_mu_qkv_rope_bcast_fwd")
        return q, k, v
    with nat.launch_region("mu_qkv", x.device, M=B * S, H=H, N=N, mu=mu2 is not None):
        nat.check(nat.lib().cdx_mu_qkv_rope_fwd(
            x2.data_ptr(), ldx, nat.ptr(mu2), ldmu, wx_ptr, wmu_ptr, ldw, B, S, H, nq, nkv, hd,
            nat.ptr(q_norm_w), nat.ptr(k_norm_w), float(eps), cos_sin.data_ptr(), cos_sin.shape[0], pos0,
            q.data_ptr(), k.data_ptr(), v.data_ptr(), vt_ld, nat.stream_of(x)), "cdx_mu_qkv_rope_fwd")
    return q, k, v


def causal_attention(q: torch.Tensor, k: torch.Tensor, vt: torch.Tensor, scale: Optional[float] = None
                     ) -> torch.Tensor:
    """softmax(q k^T * scale, top-left causal) v for GQA heads (cdx_attention_fwd).

    q [B, nq, S, D], k [B, nkv, S, D], vt = V in the transposed layout
    [B, nkv, D, vt_ld] (to_vt_layout / mu_qkv_rope(v_transposed=True)).  Returns the
    merged [B, S, nq * D] that o_proj consumes.  Equals
    F.scaled_dot_product_attention(q, k.repeat_interleave(nq // nkv, 1),
    v.repeat_interleave(nq // nkv, 1), is_causal=True) (core/attention.py:163-181)."""
    nat.require_device(q, k, vt, what="causal_attention")
    B, nq, S, D = q.shape
    nkv = k.shape[1]
    if k.shape != (B, nkv, S, D) or vt.shape[:3] != (B, nkv, D) or vt.shape[3] < S:
        raise ValueError("causal_attention: q/k/vt shapes do not match")
    if not (q.is_contiguous() and k.is_contiguous() and vt.is_contiguous()):
        raise ValueError("causal_attention: q, k and vt must be contiguous")
    scale = D ** -0.5 if scale is None else scale
    out = torch.empty(B, S, nq * D, dtype=q.dtype, device=q.device)
    with nat.launch_region("attention", q.device, B=B, S=S, nq=nq, D=D):
        nat.check(nat.lib().cdx_attention_fwd(q.data_ptr(), k.data_ptr(), vt.data_ptr(), B, S, nq, nkv, D,
                                              vt.shape[3], float(scale), out.data_ptr(), nat.stream_of(q)),
                  "cdx_attention_fwd")
    return out


# Queries up to which cdx_qkv_cache_fwd can run the attention itself (keys all cached).
_ATTEND_ROWS = 16


def qkv_cache(x: torch.Tensor, mu: Optional[torch.Tensor], w_x: torch.Tensor, w_mu: torch.Tensor, H: int, nq: int,
              nkv: int, hd: int, q_norm_w: Optional[torch.Tensor], k_norm_w: Optional[torch.Tensor], eps: float,
              cos_sin: torch.Tensor, past: Optional[Tuple[torch.Tensor, torch.Tensor]] = None
              ) -> Tuple[Optional[torch.Tensor], Optional[torch.Tensor], torch.Tensor, torch.Tensor]:
    """(q, attention, k, v) of x [B, S, H] (cdx_qkv_cache_fwd): the projection, QK norm and
    RoPE at positions past .. past + S - 1, and the cache with the new rows appended
    (k, v [B, nkv, past + S, hd]).  For a few queries whose keys are all cached the kernel
    runs the causal attention too and q is None; otherwise attention is None and q is
    [B, nq, S, hd].  past: contiguous k and v of [B, nkv, past, hd] (its first two items, so
    also one stacked tensor), or None."""
    pk, pv = (past[0], past[1]) if past is not None else (None, None)
    nat.require_device(x, mu, w_x, w_mu, q_norm_w, k_norm_w, pk, pv, what="qkv_cache")
    _check_widths(x, mu, H, "qkv_cache")
    B, S, _ = x.shape
    if w_x.shape[0] != (nq + 2 * nkv) * hd or (pk is not None and not (
            pk.shape == pv.shape == (B, nkv, pk.shape[2], hd) and pk.is_contiguous() and pv.is_contiguous())):
        raise ValueError(f"qkv_cache: weight {tuple(w_x.shape)} or cache does not match {nq} + 2 x {nkv} heads of {hd}")
    x2, ldx = _rows_view(x, H)
    if ldx == 0:
        x2, ldx = x.contiguous(), H
    mu2, ldmu = None, 0
    if mu is not None:
        mu2, ldmu = _rows_view(mu.expand(B, S, H) if mu.shape[:-1] != (B, S) else mu, H)
    wx_ptr, wmu_ptr, ldw = _weight_sources(w_x, w_mu, mu2, H, "qkv_cache")
    if q_norm_w is not None:
        q_norm_w = q_norm_w.to(x.dtype).contiguous()
        k_norm_w = k_norm_w.to(x.dtype).contiguous()
    P = pk.shape[2] if pk is not None else 0
    attend = S <= _ATTEND_ROWS and P >= S
    new = lambda *shape: torch.empty(shape, dtype=x.dtype, device=x.device)  # noqa: E731
    q = None if attend else new(B, nq, S, hd)
    attn = new(B, S, nq * hd) if attend else None
    k, v = new(B, nkv, P + S, hd), new(B, nkv, P + S, hd)
    lib = nat.lib()
    ws = lib.cdx_qkv_cache_workspace_bytes(B, S, nq, nkv, hd)
    work = torch.empty(ws, dtype=torch.uint8, device=x.device)
    with nat.launch_region("mu_qkv", x.device, M=B * S, H=H, N=(nq + 2 * nkv) * hd, mu=mu is not None):
        nat.check(lib.cdx_qkv_cache_fwd(
            x2.data_ptr(), ldx, nat.ptr(mu2), ldmu, wx_ptr, wmu_ptr, ldw, B, S, H, nq, nkv, hd, nat.ptr(q_norm_w),
            nat.ptr(k_norm_w), float(eps), cos_sin.data_ptr(), cos_sin.shape[0], nat.ptr(pk), nat.ptr(pv), P,
            nat.ptr(q), k.data_ptr(), v.data_ptr(), nat.ptr(attn), hd ** -0.5, work.data_ptr(), ws,
            nat.stream_of(x)), "cdx_qkv_cache_fwd")
    return q, attn, k, v


def cache_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """softmax(q k^T / sqrt(D), top-left causal) v merged to [B, S, nq * D], for q
    [B, nq, S, D] and a cache k, v [B, nkv, rows >= S, D] (contiguous, D a multiple of 8 up
    to 128): only the first S keys are visible to any query and read
    (cdx_vt_pack, cdx_attention_cache_fwd)."""
    nat.require_device(q, k, v, what="cache_attention")
    B, nq, S, D = q.shape
    nkv, rows = k.shape[1], k.shape[2]
    if k.shape != (B, nkv, rows, D) or v.shape != k.shape or rows < S:
        raise ValueError("cache_attention: q/k/v shapes do not match")
    if not (q.is_contiguous() and k.is_contiguous() and v.is_contiguous()):
        raise ValueError("cache_attention: q, k and v must be contiguous")
    vt_ld = vt_ld_for(S)
    vt = torch.empty(B, nkv, D, vt_ld, dtype=q.dtype, device=q.device)
    out = torch.empty(B, S, nq * D, dtype=q.dtype, device=q.device)
    lib, stream = nat.lib(), nat.stream_of(q)
    with nat.launch_region("attention", q.device, B=B, S=S, nq=nq, D=D):
        nat.check(lib.cdx_vt_pack(v.data_ptr(), B * nkv, rows, S, D, vt.data_ptr(), vt_ld, stream), "cdx_vt_pack")
        nat.check(lib.cdx_attention_cache_fwd(q.data_ptr(), k.data_ptr(), vt.data_ptr(), B, S, rows, nq, nkv, D, vt_ld,
                                              D ** -0.5, out.data_ptr(), stream), "cdx_attention_cache_fwd")
    return out


def fused_mu_qkv_projection(x: torch.Tensor, mu: Optional[torch.Tensor], wq: torch.Tensor,
                            wk: torch.Tensor, wv: torch.Tensor, mu_wq: torch.Tensor,
                            mu_wk: torch.Tensor, mu_wv: torch.Tensor
                            ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """q = x@wq + mu@mu_wq (k, v alike) with weights [in, out]; cuda/triton_mu_qkv.py:195-283.
    Returns [B, S, q_dim], [B, S, kv_dim], [B, S, kv_dim] (column views of one buffer)."""
    forward_only("fused_mu_qkv_projection", x, mu, wq, wk, wv, mu_wq, mu_wk, mu_wv)
    H = x.shape[-1]
    q_dim, kv_dim = wq.shape[1], wk.shape[1]
    w_x = torch.cat([wq, wk, wv], dim=1)
    if mu is not None:
        w_mu = torch.cat([mu_wq, mu_wk, mu_wv], dim=1)
        w_pack = torch.cat([w_x, w_mu], dim=0).t().contiguous()
    else:
        w_pack = w_x.t().contiguous()
    out = mu_qkv_project(x, mu, w_pack, H)
    return (out[..., :q_dim], out[..., q_dim:q_dim + kv_dim], out[..., q_dim + kv_dim:])


class FusedMuQKVProjection(nn.Module):
    """Module form of the fused projection; cuda/triton_mu_qkv.py:336-394."""

    def __init__(self, hidden_size: int, num_attention_heads: int, num_key_value_heads: int):
        super().__init__()
        self.hidden_size = hidden_size
        self.num_heads = num_attention_heads
        self.num_kv_heads = num_key_value_heads
        self.head_dim = hidden_size // num_attention_heads
        self.q_dim = num_attention_heads * self.head_dim
        self.kv_dim = num_key_value_heads * self.head_dim
        self.q_proj = nn.Linear(hidden_size, self.q_dim, bias=False)
        self.k_proj = nn.Linear(hidden_size, self.kv_dim, bias=False)
        self.v_proj = nn.Linear(hidden_size, self.kv_dim, bias=False)
        self.mu_to_q = nn.Linear(hidden_size, self.q_dim, bias=False)
        self.mu_to_k = nn.Linear(hidden_size, self.kv_dim, bias=False)
        self.mu_to_v = nn.Linear(hidden_size, self.kv_dim, bias=False)
        self._qkv_w = QKVWeights()

    def forward(self, x: torch.Tensor, mu: Optional[torch.Tensor] = None):
        forward_only("FusedMuQKVProjection", x, mu, module=self)
        w_x, w_mu = self._qkv_w.get(self)
        out = mu_qkv_project(x, mu, w_x, self.hidden_size, w_mu=w_mu)
        return (out[..., : self.q_dim], out[..., self.q_dim: self.q_dim + self.kv_dim],
                out[..., self.q_dim + self.kv_dim:])


# The methods that the shorter paths stand in for, as the modules of their classes define them:
# dispatch and instrumentation libraries replace them, on the instance or on the class (then
# also before this import, which is why a method of another module's is not taken down).
_WRITTEN: dict = {}


def _own_method(cls: type, name: str):
    f = getattr(cls, name)
    return f if getattr(f, "__globals__", None) is vars(sys.modules[cls.__module__]) else None


def _written(*classes: type) -> None:
    _WRITTEN.update({c: _own_method(c, "forward") for c in classes})


_MODULE_CALL = _own_method(nn.Module, "__call__")
_written(nn.Linear, nn.RMSNorm, RotaryEmbedding)


def _as_written(m: nn.Module) -> bool:
    """Whether calling m runs the forward its class was written with and nothing else: no hook,
    its own or a global one, and no forward set on the instance or the class.  (Of the classes
    given to _written; False for any other.)"""
    cls = type(m)
    return (cls.forward is _WRITTEN.get(cls) and cls.__call__ is _MODULE_CALL
            and not (m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__
                     or nn.modules.module._has_any_global_hook()))


def _plain_norm(m: nn.Module, D: int) -> bool:
    """Whether m is an unhooked nn.RMSNorm over D values with a weight and an eps."""
    return (type(m) is nn.RMSNorm and m.weight is not None and m.weight.shape == (D,) and m.eps is not None
            and _as_written(m))


def _plain_linear(m: nn.Module) -> bool:
    """Whether calling m is exactly F.linear(x, m.weight): no subclass, bias, hook or autocast."""
    return (type(m) is nn.Linear and m.bias is None and type(m.weight) is nn.Parameter
            and _as_written(m) and not torch.is_autocast_enabled())


class QKVWeights:
    """The kernel operands W_x = [Wq; Wk; Wv] and W_mu = [Wmu_q; Wmu_k; Wmu_v] of one
    module, side by side in one [N, 2H] buffer (row n = [W_x[n] | W_mu[n]], the
    reference's torch.cat([q_proj.weight, mu_to_q.weight], dim=1) for each of q, k, v)
    whose column halves the six Linear weights are views of.

    A write to a weight (in place, through ``.data``, by load_state_dict) therefore
    lands in the operand the kernel reads; nothing is cached that could go stale.
    When a weight is no longer its view (the module was moved or cast, a Parameter was
    replaced), ``get`` copies the current weights into a new buffer and re-points them
    at it.  The buffer is made outside inference mode, so that the weights stay
    writable after a forward run under torch.inference_mode()."""

    def __init__(self):
        self.buf: Optional[torch.Tensor] = None
        self.ptrs = None

    @staticmethod
    def _linears(m):
        return (m.q_proj, m.k_proj, m.v_proj, m.mu_to_q, m.mu_to_k, m.mu_to_v)

    _NAMES = ("q_proj", "k_proj", "v_proj", "mu_to_q", "mu_to_k", "mu_to_v")

    def buffer(self, m) -> torch.Tensor:
        """The [N, 2H] buffer, holding m's current weights."""
        mods = m._modules
        try:  # lin.weight of every projection, without nn.Module's attribute search
            ws = [mods[n]._parameters["weight"] for n in self._NAMES]
        except (KeyError, AttributeError):
            ws = [lin.weight for lin in self._linears(m)]
        if self.buf is None or [w.data_ptr() for w in ws] != self.ptrs:
            self._bind(ws, m.hidden_size)
        return self.buf

    def get(self, m) -> Tuple[torch.Tensor, torch.Tensor]:
        buf, H = self.buffer(m), m.hidden_size
        return buf[:, :H], buf[:, H:]

    def _bind(self, ws, H: int) -> None:
        dt, dev = ws[0].dtype, ws[0].device
        if any(w.dtype != dt or w.device != dev or w.dim() != 2 or w.shape[1] != H for w in ws):
            raise ValueError("ComplexityAttention: the q/k/v and mu_to_q/k/v weights must share one dtype "
                             f"and device and be [out, {H}]")
        xs, mus = ws[:3], ws[3:]
        if [w.shape[0] for w in xs] != [w.shape[0] for w in mus]:
            raise ValueError("ComplexityAttention: mu_to_q/k/v must have the shapes of q/k/v_proj")
        N = sum(w.shape[0] for w in xs)
        with torch.inference_mode(False), torch.no_grad():
            buf = torch.empty(N, 2 * H, dtype=dt, device=dev)
            r = 0
            for wx, wm in zip(xs, mus):
                n = wx.shape[0]
                buf[r:r + n, :H].copy_(wx)
                buf[r:r + n, H:].copy_(wm)
                wx.data = buf[r:r + n, :H]
                wm.data = buf[r:r + n, H:]
                r += n
        self.buf = buf
        self.ptrs = [w.data_ptr() for w in ws]


class ComplexityAttention(nn.Module):
    """GQA attention with mu guidance and QK normalisation; core/attention.py:33-181."""

    def __init__(self, hidden_size: int, num_attention_heads: int, num_key_value_heads: int,
                 max_position_embeddings: int = 2048, rope_theta: float = 10000.0,
                 attention_dropout: float = 0.0, use_qk_norm: bool = True):
        super().__init__()
        self.hidden_size = hidden_size
        self.num_heads = num_attention_heads
        self.num_kv_heads = num_key_value_heads
        self.head_dim = hidden_size // num_attention_heads
        self.num_kv_groups = num_attention_heads // num_key_value_heads
        if self.head_dim * num_attention_heads != hidden_size:
            raise ValueError("hidden_size must be divisible by num_attention_heads")
        if num_attention_heads % num_key_value_heads != 0:
            raise ValueError("num_attention_heads must be a multiple of num_key_value_heads")
        q_dim = num_attention_heads * self.head_dim
        kv_dim = num_key_value_heads * self.head_dim
        # Registration order matters for seeded init parity (one draw per Linear).
        self.q_proj = nn.Linear(hidden_size, q_dim, bias=False)
        self.k_proj = nn.Linear(hidden_size, kv_dim, bias=False)
        self.v_proj = nn.Linear(hidden_size, kv_dim, bias=False)
        self.o_proj = nn.Linear(q_dim, hidden_size, bias=False)
        self.mu_to_q = nn.Linear(hidden_size, q_dim, bias=False)
        self.mu_to_k = nn.Linear(hidden_size, kv_dim, bias=False)
        self.mu_to_v = nn.Linear(hidden_size, kv_dim, bias=False)
        self.use_qk_norm = use_qk_norm
        if use_qk_norm:
            self.q_norm = nn.RMSNorm(self.head_dim, eps=1e-6)
            self.k_norm = nn.RMSNorm(self.head_dim, eps=1e-6)
        self.rotary_emb = RotaryEmbedding(self.head_dim, max_seq_len=max_position_embeddings, theta=rope_theta)
        self.attention_dropout = attention_dropout
        self._qkv_w = QKVWeights()

    def qkv_weights(self) -> Tuple[torch.Tensor, torch.Tensor]:
        """(W_x, W_mu), each [Nq*D + 2*Nkv*D, H]: the two column halves of the [N, 2H]
        buffer the six projection weights are views of, i.e. exactly what the kernels read."""
        return self._qkv_w.get(self)

    def project_qkv(self, hidden_states: torch.Tensor, mu_prev: Optional[torch.Tensor]) -> torch.Tensor:
        """Packed [.., Nq*D + 2*Nkv*D] projection through the gfx950 MFMA kernel."""
        w_x, w_mu = self.qkv_weights()
        return mu_qkv_project(hidden_states, mu_prev, w_x, self.hidden_size, w_mu=w_mu)

    @property
    def fused_prologue(self) -> bool:
        """Whether QK-norm + RoPE run inside the projection kernel (cdx_mu_qkv_rope_fwd
        handles head dims 32, 64 and 128 and H a multiple of 64)."""
        return self.head_dim in (32, 64, 128) and self.hidden_size % 64 == 0

    @property
    def other_head_dim(self) -> bool:
        """Whether the heads run on the kernels through cdx_qkv_cache_fwd alone: a head dim
        that is a multiple of 8 up to 128 other than 32, 64 and 128, with the module's own
        norms and rotary tables in place."""
        D = self.head_dim
        return (D not in (32, 64, 128) and D % 8 == 0 and D <= 128 and self.hidden_size % 64 == 0
                and type(self.rotary_emb) is RotaryEmbedding and _as_written(self.rotary_emb)
                and (not self.use_qk_norm or (_plain_norm(self.q_norm, D) and _plain_norm(self.k_norm, D)
                                              and self.q_norm.eps == self.k_norm.eps)))

    def _cache_fits(self, past, x: torch.Tensor) -> bool:
        """Whether the kernels take this KV cache (None: a prompt): plain contiguous tensors of
        the module's shape, and counts within cdx_qkv_cache_fwd's 31 bits (16-byte pieces of
        the caches, (token, head) rows).  Any other goes through torch.cat and SDPA."""
        B, S, _ = x.shape
        D, nq, nkv = self.head_dim, self.num_heads, self.num_kv_heads
        rows = S + (past[0].shape[2] if past is not None else 0)
        if 2 * B * nkv * rows * D // 8 >= 2 ** 31 or B * S * (nq + 2 * nkv) >= 2 ** 31:
            return False
        if past is None:
            return True
        k, v = past[0], past[1]
        return (k.dim() == 4 and k.shape == (B, nkv, k.shape[2], D) and v.shape == k.shape and k.shape[2] > 0
                and all(t.dtype == x.dtype and t.device == x.device and t.is_contiguous() and t.data_ptr() % 16 == 0
                        and not (t.requires_grad and torch.is_grad_enabled()) for t in (k, v)))

    def _cache_attention(self, x: torch.Tensor, mu: Optional[torch.Tensor], past, use_cache: bool,
                         residual: Optional[torch.Tensor]):
        """The attention (no mask, no dropout) with a KV cache, of a few rows or at another
        head dim, on the kernels."""
        nat.require_device(x, what="ComplexityAttention")
        B, S, _ = x.shape
        H, D, nq, nkv = self.hidden_size, self.head_dim, self.num_heads, self.num_kv_heads
        past_len = past[0].shape[2] if past is not None else 0
        w_x, w_mu = self.qkv_weights()
        table = self.rotary_emb.cos_sin_table(past_len + S, x.device)
        qn = (self.q_norm.weight, self.k_norm.weight) if self.use_qk_norm else (None, None)
        eps = self.q_norm.eps if self.use_qk_norm else 0.0
        if D not in (32, 64, 128) or few_rows(B * S, (nq + 2 * nkv) * D):
            # A few rows: the fused epilogue needs whole heads in a tile, i.e. a handful of
            # blocks (one 1B layer, 4 rows: 78 us on 16 CUs; product and pass here 17 us).
            q, attn, k, v = qkv_cache(x, mu, w_x, w_mu, H, nq, nkv, D, *qn, eps, table, past)
            if attn is None:
                attn = cache_attention(q, k, v)
        else:
            q, k, v = mu_qkv_rope(x, mu, w_x, H, nq, nkv, D, *qn, eps, table, past_len, w_mu=w_mu)
            if past is not None:
                k, v = torch.cat([past[0], k], dim=2), torch.cat([past[1], v], dim=2)
            attn = cache_attention(q, k, v)
        return self._out_proj(attn, residual), (k, v) if use_cache else None

    def _out_proj(self, attn: torch.Tensor, residual: Optional[torch.Tensor]) -> torch.Tensor:
        """o_proj(attn), or with ``residual``: residual + o_proj(attn) written into residual
        (one GEMM with beta = 1, the block's residual add of core/layer.py:174).  o_proj is
        not one of the path's three pieces; hipBLASLt's beta = 1 GEMM ran the 1B forward
        0.8% faster than the tile engine's o_proj + residual kernel (linear_residual_), so
        the model keeps it.  The few rows of a generation step run on the kernels for few
        rows instead (4 x 2048 x 2048: 4.4 us, the library's 8.4 us), unless o_proj is
        more than a plain Linear."""
        rows = attn.shape[0] * attn.shape[1]
        own = rows <= 64 and _plain_linear(self.o_proj)
        if own:
            w = self.o_proj.weight
            own = (few_rows(rows, w.shape[0]) and w.dtype == attn.dtype and w.is_contiguous()
                   and w.data_ptr() % 16 == 0 and w.shape[0] % 8 == 0 and w.shape[1] % 64 == 0)
        if residual is None:
            return linear(attn, w) if own else self.o_proj(attn)
        if residual.shape[:-1] != attn.shape[:-1] or not residual.is_contiguous():
            raise ValueError("ComplexityAttention: residual must be contiguous and match the input rows")
        if own and residual.dtype == attn.dtype and residual.data_ptr() % 16 == 0:
            return linear_accumulate_(attn, w, residual)
        residual.view(-1, residual.shape[-1]).addmm_(attn.reshape(-1, attn.shape[-1]), self.o_proj.weight.t())
        return residual

    def forward(self, hidden_states: torch.Tensor, attention_mask: Optional[torch.Tensor] = None,
                past_key_value: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
                use_cache: bool = False, mu_prev: Optional[torch.Tensor] = None,
                residual: Optional[torch.Tensor] = None):
        """Returns (o_proj(attention), new_kv); with ``residual`` (the block input h,
        contiguous) the output is added to it in place and residual is returned."""
        forward_only("ComplexityAttention", hidden_states, mu_prev, residual, module=self)
        B, S, _ = hidden_states.shape
        D = self.head_dim
        past_len = past_key_value[0].shape[2] if past_key_value is not None else 0
        if attention_mask is None and not (self.training and self.attention_dropout > 0):
            cached = past_key_value is not None or use_cache
            fused = self.fused_prologue
            fast = nat.host()
            if fast is not None and (fused or self.other_head_dim) and hidden_states.is_cuda:
                qn = (self.q_norm.weight, self.k_norm.weight) if self.use_qk_norm else (None, None)
                pk, pv = (past_key_value[0], past_key_value[1]) if past_key_value is not None else (None, None)
                done = fast.attention(hidden_states, mu_prev, self._qkv_w.buffer(self), self.num_heads,
                                      self.num_kv_heads, D, *qn, self.q_norm.eps if self.use_qk_norm else 0.0,
                                      self.rotary_emb.cos_sin_table(past_len + S, hidden_states.device), pk, pv,
                                      use_cache)
                if done is not None:
                    attn, k, v = done
                    return self._out_proj(attn, residual), (k, v) if use_cache else None
            if fused and not cached and not few_rows(B * S, (self.num_heads + 2 * self.num_kv_heads) * D):
                # Fused projection (V written transposed) and the causal GQA kernel, whose
                # output is already merged over heads.
                w_x, w_mu = self.qkv_weights()
                table = self.rotary_emb.cos_sin_table(S, hidden_states.device)
                qn = (self.q_norm.weight, self.k_norm.weight) if self.use_qk_norm else (None, None)
                eps = self.q_norm.eps if self.use_qk_norm else 0.0
                q, k, vt = mu_qkv_rope(hidden_states, mu_prev, w_x, self.hidden_size, self.num_heads,
                                       self.num_kv_heads, D, qn[0], qn[1], eps, table, 0, v_transposed=True,
                                       w_mu=w_mu)
                return self._out_proj(causal_attention(q, k, vt), residual), None
            if B * S > 0 and (fused or self.other_head_dim) and self._cache_fits(past_key_value, hidden_states):
                return self._cache_attention(hidden_states, mu_prev, past_key_value, use_cache, residual)
        if self.fused_prologue:
            # Projection, head split, QK RMSNorm and RoPE in one kernel (attention.py:120-155).
            w_x, w_mu = self.qkv_weights()
            table = self.rotary_emb.cos_sin_table(past_len + S, hidden_states.device)
            qn = (self.q_norm.weight, self.k_norm.weight) if self.use_qk_norm else (None, None)
            eps = self.q_norm.eps if self.use_qk_norm else 0.0
            q, k, v = mu_qkv_rope(hidden_states, mu_prev, w_x, self.hidden_size, self.num_heads,
                                  self.num_kv_heads, D, qn[0], qn[1], eps, table, past_len, w_mu=w_mu)
        else:
            q_dim, kv_dim = self.num_heads * D, self.num_kv_heads * D
            qkv = self.project_qkv(hidden_states, mu_prev)
            q = qkv[..., :q_dim].view(B, S, self.num_heads, D).transpose(1, 2)
            k = qkv[..., q_dim:q_dim + kv_dim].view(B, S, self.num_kv_heads, D).transpose(1, 2)
            v = qkv[..., q_dim + kv_dim:].view(B, S, self.num_kv_heads, D).transpose(1, 2)
            if self.use_qk_norm:
                q = self.q_norm(q)
                k = self.k_norm(k)
            kv_seq_len = S + past_len
            cos, sin = self.rotary_emb(kv_seq_len)
            cos = cos.to(q.device, dtype=q.dtype)
            sin = sin.to(q.device, dtype=q.dtype)
            if past_key_value is not None:
                cos, sin = cos[kv_seq_len - S:], sin[kv_seq_len - S:]
            q, k = apply_rotary_pos_emb(q, k, cos, sin)
        if past_key_value is not None:
            k = torch.cat([past_key_value[0], k], dim=2)
            v = torch.cat([past_key_value[1], v], dim=2)
        new_kv = (k, v) if use_cache else None
        k = k.repeat_interleave(self.num_kv_groups, dim=1)
        v = v.repeat_interleave(self.num_kv_groups, dim=1)
        # Same SDPA call as the reference, including is_causal=(mask is None).
        attn = F.scaled_dot_product_attention(
            q, k, v, attn_mask=attention_mask,
            dropout_p=self.attention_dropout if self.training else 0.0,
            is_causal=attention_mask is None)
        attn = attn.transpose(1, 2).contiguous().view(B, S, -1)
        return self._out_proj(attn, residual), new_kv


MuGuidedAttention = ComplexityAttention
_written(ComplexityAttention)

__all__ = ["ComplexityAttention", "MuGuidedAttention", "FusedMuQKVProjection", "fused_mu_qkv_projection",
           "mu_qkv_project", "mu_qkv_rope", "causal_attention", "to_vt_layout", "vt_columns", "QKVWeights"]
