"""ComplexityAttention with a KV cache, and at head dims other than 32, 64 and 128, on the
kernels (cdx_qkv_cache_fwd, cdx_vt_pack, cdx_attention_cache_fwd) against a float64
restatement of core/attention.py:120-181: projection, QK norm, RoPE at the cached position,
the extended cache, and causal attention aligned at the top left."""

from __future__ import annotations

import math

import pytest
import torch

from _metrics import assert_close_bf16, errors

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _rope(x, pos0):
    D, S = x.shape[-1], x.shape[-2]
    inv = 10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64) / D)
    a = torch.outer(torch.arange(pos0, pos0 + S, dtype=torch.float64), inv)
    x1, x2 = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([x1 * a.cos() - x2 * a.sin(), x2 * a.cos() + x1 * a.sin()], -1)


def _reference(m, x, mu, past):
    d = lambda t: t.detach().double().cpu()  # noqa: E731
    B, S, _ = x.shape
    D, nq, nkv = m.head_dim, m.num_heads, m.num_kv_heads

    def project(w, w_mu, heads, norm=None):
        y = d(x) @ d(w.weight).t() + (0 if mu is None else d(mu) @ d(w_mu.weight).t())
        y = y.view(B, S, heads, D).transpose(1, 2)
        return y if norm is None else y * torch.rsqrt(y.square().mean(-1, keepdim=True) + norm.eps) * d(norm.weight)

    norms = (m.q_norm, m.k_norm) if m.use_qk_norm else (None, None)
    P = past[0].shape[2] if past is not None else 0
    q = _rope(project(m.q_proj, m.mu_to_q, nq, norms[0]), P)
    k = _rope(project(m.k_proj, m.mu_to_k, nkv, norms[1]), P)
    v = project(m.v_proj, m.mu_to_v, nkv)
    if past is not None:
        k, v = torch.cat([d(past[0]), k], 2), torch.cat([d(past[1]), v], 2)
    kr, vr = (t[:, :, :S].repeat_interleave(nq // nkv, 1) for t in (k, v))
    s = (q @ kr.transpose(-1, -2)) / math.sqrt(D)
    s = s.masked_fill(~torch.ones(S, S, dtype=torch.bool).tril(), -math.inf).softmax(-1)
    return (s @ vr).transpose(1, 2).reshape(B, S, -1) @ d(m.o_proj.weight).t(), k, v


def _module(cdx, nq, nkv, D, qk_norm=True, seed=0):
    torch.manual_seed(seed)
    m = cdx.ComplexityAttention(nq * D, nq, nkv, use_qk_norm=qk_norm).to(bf16).cuda().eval()
    if qk_norm:
        with torch.no_grad():
            m.q_norm.weight.normal_(1, 0.1)
            m.k_norm.weight.normal_(1, 0.1)
    return m


@pytest.mark.parametrize("D,nq,nkv,B,S,past,mu,qk_norm", [
    (128, 8, 4, 3, 1, 300, "rows", True), (64, 12, 4, 1, 1, 1, "rows", True),    # a step
    (64, 4, 2, 2, 16, 16, "row", True), (64, 4, 1, 2, 17, 40, "rows", False),    # the attending pass's edge
    (64, 4, 2, 2, 3, 2, "rows", True), (32, 4, 4, 4, 16, 0, None, True),         # keys among the new tokens
    (128, 4, 2, 2, 200, 0, "rows", True), (64, 4, 2, 1, 130, 70, "rows", True),  # prompts: fused projection
    (80, 16, 4, 2, 77, 0, "rows", True), (80, 4, 4, 3, 1, 129, "row", True),     # other head dims
    (40, 8, 4, 1, 200, 33, "rows", True), (8, 8, 8, 2, 65, 0, "rows", True), (24, 8, 2, 1, 64, 0, "rows", False),
    (48, 4, 1, 2, 63, 5, "rows", True), (56, 8, 4, 1, 129, 0, None, True), (96, 2, 1, 1, 128, 0, "rows", True),
    (104, 8, 1, 1, 70, 0, "rows", True), (120, 8, 8, 1, 257, 0, "rows", True),
])
def test_attention_with_a_cache(cdx, D, nq, nkv, B, S, past, mu, qk_norm):
    print(f"kv cache D={D} heads={nq}/{nkv} B={B} S={S} past={past} mu={mu} qk_norm={qk_norm}", flush=True)
    m = _module(cdx, nq, nkv, D, qk_norm, seed=D + S)
    H = nq * D
    g = torch.Generator().manual_seed(S + past)
    new = lambda *s: torch.randn(*s, generator=g).to(bf16).cuda()  # noqa: E731
    x = new(B, S, H)
    mus = None if mu is None else (new(B, S, H) if mu == "rows" else new(1, 1, H).expand(B, S, H))
    kv = (new(B, nkv, past, D), new(B, nkv, past, D)) if past else None
    with torch.no_grad():
        out, (k, v) = m(x, mu_prev=mus, past_key_value=kv, use_cache=True)
        plain, none = m(x, mu_prev=mus, past_key_value=kv)
        h = new(B, S, H)
        added, _ = m(x, mu_prev=mus, past_key_value=kv, use_cache=True, residual=h.clone())
    ref, rk, rv = _reference(m, x, mus, kv)
    assert none is None
    assert_close_bf16(out, ref, "out")
    assert_close_bf16(plain, ref, "out, no cache kept")
    assert_close_bf16(added, h.double().cpu() + ref, "residual")
    if D in (32, 64, 128) or B * S <= 64:
        assert_close_bf16(k, rk, "k")
    else:
        # The projection is rounded to bf16 before the norm, then the result: two roundings
        # of at most 2^-9 of a value each.
        e = errors(k, rk)
        assert e["rel_rms"] <= 2 * 2.0 ** -9 and e["max_rel"] <= 2.0 ** -7, f"k: {e}"
    assert_close_bf16(v, rv, "v")
    if past:
        assert torch.equal(k[:, :, :past], kv[0]) and torch.equal(v[:, :, :past], kv[1])


def test_caches_the_kernels_do_not_take(cdx):
    """A strided cache, and a mask, keep the torch.cat and SDPA path; the strided cache gives
    what its contiguous copy gives."""
    print("kv cache: strided, masked", flush=True)
    m = _module(cdx, 4, 2, 64)
    x = torch.randn(2, 3, 256, device="cuda").to(bf16)
    kv = tuple(torch.randn(2, 9, 2, 64, device="cuda").to(bf16).transpose(1, 2) for _ in range(2))
    with torch.no_grad():
        a, (ka, va) = m(x, past_key_value=kv, use_cache=True)
        b, (kb, vb) = m(x, past_key_value=tuple(t.contiguous() for t in kv), use_cache=True)
        every = torch.ones(3, 12, dtype=torch.bool, device="cuda")
        c, (kc, _) = m(x, past_key_value=kv, use_cache=True, attention_mask=every)
    assert_close_bf16(a, b.float(), "strided cache")
    assert_close_bf16(ka, kb.float(), "strided cache k")
    assert_close_bf16(va, vb.float(), "strided cache v")
    assert torch.equal(kc, ka) and not torch.equal(c, a)


def test_vt_pack_matches_the_layout(cdx):
    from complexity_deep import _native as nat
    from complexity_deep.attention import to_vt_layout, vt_ld_for
    print("vt_pack", flush=True)
    for D, S, rows in ((128, 64, 64), (80, 65, 70), (8, 1, 300), (40, 63, 63)):
        v = torch.randn(2, 3, rows, D, device="cuda").to(bf16)
        vt = torch.full((2, 3, D, vt_ld_for(S)), float("nan"), dtype=bf16, device="cuda")
        nat.check(nat.lib().cdx_vt_pack(v.data_ptr(), 6, rows, S, D, vt.data_ptr(), vt.shape[-1], nat.stream_of(v)),
                  "cdx_vt_pack")
        assert torch.equal(vt, to_vt_layout(v[:, :, :S].contiguous())), (D, S, rows)


def test_vt_pack_of_more_slabs_than_a_grid_axis(cdx):
    """Batch x KV heads past 65535, the limit of a grid's second axis."""
    from complexity_deep import _native as nat
    from complexity_deep.attention import to_vt_layout, vt_ld_for
    print("vt_pack, 65537 slabs", flush=True)
    slabs, S, rows, D = 65537, 2, 3, 8
    v = torch.randn(1, slabs, rows, D, device="cuda").to(bf16)
    vt = torch.full((1, slabs, D, vt_ld_for(S)), float("nan"), dtype=bf16, device="cuda")
    nat.check(nat.lib().cdx_vt_pack(v.data_ptr(), slabs, rows, S, D, vt.data_ptr(), vt.shape[-1], nat.stream_of(v)),
              "cdx_vt_pack")
    assert torch.equal(vt, to_vt_layout(v[:, :, :S].contiguous()))


def test_a_score_of_minus_infinity_in_a_step(cdx):
    """An infinite value in a cached key gives scores of -inf (no weight: the row stays finite
    while another key has one) or +inf (NaN), as softmax does."""
    print("kv cache: infinite keys", flush=True)
    m = _module(cdx, 1, 1, 64, seed=5)
    g = torch.Generator().manual_seed(6)
    new = lambda *s: torch.randn(*s, generator=g).to(bf16).cuda()  # noqa: E731
    B, S, past = 12, 5, 9  # (at most 64 rows: the pass over the cache attends itself)
    x, kv = new(B, S, 64), [new(B, 1, past, 64), new(B, 1, past, 64)]
    kv[0][:, :, 0, 3] = math.inf
    kv[0][::2, :, 2, 3] = math.inf
    with torch.no_grad():
        out, _ = m(x, past_key_value=kv, use_cache=True)
    ref, _, _ = _reference(m, x, None, kv)
    finite = torch.isfinite(ref).all(-1)
    assert 0 < int(finite.sum()) < B * S and bool(finite[1::2, 1:].any())
    assert torch.equal(torch.isfinite(out).all(-1).cpu(), finite)
    assert_close_bf16(out.cpu()[finite], ref[finite], "finite rows")
