"""The kernels for products of a few rows (M <= 64, the linear layers and the MoE of a
generation step) against fp32 references, at the edges of their row groups (16, 32, 64
rows; 65 is the tile engine's), with column counts that end inside a block, K shares that
leave waves without work, and both K sources."""

from __future__ import annotations

import pytest
import torch

from _metrics import assert_close_bf16

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _data(seed, *shape, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(bf16).cuda()


@pytest.mark.parametrize("M,K,N", [(1, 64, 8), (1, 2048, 4096), (8, 576, 1003), (8, 704, 12296), (9, 704, 12296), (15, 320, 1003), (16, 576, 24), (17, 768, 10000),
                                   (32, 2048, 2056), (33, 1280, 200), (64, 704, 12296), (64, 64, 40), (65, 704, 40)])
def test_products_of_a_few_rows(cdx, M, K, N):
    """linear, its residual form, mu-QKV (two sources, and a broadcast mu) and mu guidance.
    The residual form adds the rounded product: linear() plus torch's bf16 add, exactly."""
    from complexity_deep.attention import mu_qkv_project
    from complexity_deep.layer import mu_guidance
    from complexity_deep.linear import linear, linear_residual_
    print(f"few rows M={M} K={K} N={N}", flush=True)
    x, w = _data(M, M, K), _data(N, N, K, scale=K ** -0.5)
    prod = linear(x, w)
    assert_close_bf16(prod, x.float() @ w.float().t(), "linear")
    wide = _data(5, M, 2 * K)  # rows at a stride of 2K
    if N % 8 == 0:
        r = _data(7, M, N)
        assert torch.equal(linear_residual_(x, w, r.clone()), r + prod)
        w2 = _data(8, N, 2 * K, scale=(2 * K) ** -0.5)
        for mu in (wide[:, K:].view(1, M, K), _data(9, 1, 1, K).expand(1, M, K)):
            got = mu_qkv_project(wide[:, :K].view(1, M, K), mu, w2, K)
            ref = wide[:, :K].float() @ w2[:, :K].float().t() + mu[0].float() @ w2[:, K:].float().t()
            assert_close_bf16(got.view(M, N), ref, "mu_qkv")
    wm, bias = _data(10, K, K, scale=K ** -0.5), _data(11, K)
    pair = torch.zeros(M, 2 * K, dtype=bf16, device="cuda")
    mu_guidance(x, wm, bias, 0.0, 2.0, -2.0, 2.0, out=pair[:, K:])
    ref = (x.float() @ wm.float().t() + bias.float().clamp(0, 2)).clamp(-2, 2)
    assert_close_bf16(pair[:, K:], ref, "mu_guidance")
    assert not bool(pair[:, :K].any())


@pytest.mark.parametrize("T,H,Ie,E,shared", [(1, 256, 176, 4, True), (3, 2048, 704, 8, True), (8, 320, 224, 16, True), (9, 320, 224, 4, False), (16, 320, 224, 4, False),
                                             (17, 1280, 864, 4, True), (33, 512, 64, 64, True), (64, 768, 512, 2, False),
                                             (64, 128, 40, 1, True)])
def test_moe_of_a_few_tokens(cdx, oracle, T, H, Ie, E, shared):
    """Experts without tokens among them; the residual form adds the rounded rows."""
    print(f"moe few tokens T={T} H={H} Ie={Ie} E={E} shared={shared}", flush=True)
    torch.manual_seed(T)
    m = cdx.TokenRoutedMLP(H, Ie * E, num_experts=E, vocab_size=500, shared_expert=shared)
    with torch.no_grad():
        m.token_to_expert.copy_(torch.randint(0, max(1, E - 1), (500,)))  # the last expert is never used
    m = m.to(bf16).cuda()
    ids = torch.randint(0, 500, (1, T))
    x, r = _data(1, 1, T, H), _data(2, 1, T, H)
    with torch.no_grad():
        got = m(x, token_ids=ids.cuda())
        added = m(x, token_ids=ids.cuda(), residual=r.clone())
    ref = oracle.token_routed_mlp(
        x.float().cpu(), ids, m.token_to_expert.cpu().numpy(), m.gate_proj_w.float().cpu(), m.up_proj_w.float().cpu(),
        m.down_proj_w.float().cpu(), *(getattr(m, n).weight.float().cpu() if shared else None
                                       for n in ("shared_gate", "shared_up", "shared_down")))
    assert_close_bf16(got, ref, "moe")
    assert torch.equal(added, r + got)


def test_segments_that_cover_part_of_the_rows(cdx):
    """persistent_swiglu_cggr over offsets that leave rows outside every segment: those rows
    stay zero."""
    print("few rows, partial segments", flush=True)
    T, H, ie, E = 40, 128, 64, 3
    x, g, u, d = _data(1, T, H), _data(2, E, H, ie, scale=0.1), _data(3, E, H, ie, scale=0.1), _data(4, E, ie, H, scale=0.1)
    offs = torch.tensor([3, 20, 20, 37], device="cuda")
    out = cdx.persistent_swiglu_cggr(x, g, u, d, offs)
    ref = torch.zeros(T, H)
    for e, (a, b) in enumerate(((3, 20), (20, 20), (20, 37))):
        t = x[a:b].float()
        ref[a:b] = ((torch.nn.functional.silu(t @ g[e].float()) * (t @ u[e].float())) @ d[e].float()).cpu()
    assert_close_bf16(out, ref, "partial segments")
    assert not bool(out[:3].any()) and not bool(out[37:].any())


@pytest.mark.parametrize("T", [2, 8, 9, 16, 31, 64])
@pytest.mark.parametrize("shared", [True, False])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_weights_that_are_not_finite_stay_with_their_expert(cdx, T, shared, bad):
    """An Inf or NaN in one expert's weights reaches that expert's tokens and no others: their
    rows have the bits that they have with finite weights."""
    print(f"few rows, {bad} in one expert, T={T} shared={shared}", flush=True)
    torch.manual_seed(T)
    H, E = 256, 4
    m = cdx.TokenRoutedMLP(H, 96 * E, num_experts=E, vocab_size=500, shared_expert=shared).to(bf16).cuda()
    ids = torch.arange(T).view(1, T) * 7 % 500
    ids[0, 1] = 1  # expert 1 has a token
    ids = ids.cuda()
    hit = m.token_to_expert[ids[0]] == 1
    x, r = _data(1, 1, T, H), _data(2, 1, T, H)
    with torch.no_grad():
        good = m(x, token_ids=ids)[0]
        added = m(x, token_ids=ids, residual=r.clone())[0]
        for name in ("down_proj_w", "gate_proj_w"):
            w = getattr(m, name).data
            keep = w[1].clone()
            w[1] = bad
            out = m(x, token_ids=ids)[0]
            out_r = m(x, token_ids=ids, residual=r.clone())[0]
            w[1] = keep
            assert bool(hit.any()) and not bool(torch.isfinite(out[hit]).any()), name
            assert torch.equal(out[~hit], good[~hit]) and torch.equal(out_r[~hit], added[~hit]), name
