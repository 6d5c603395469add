"""Products between one 128-row tile per CU and whole rounds of 256 x 256 tiles (128 x 64 and
128 x 128 tiles, one or two per CU), at the edges of the rule that picks them: the first rows
of a large product equal the product of those rows alone bit for bit (every tile form adds
along K in one order), with rows and columns that end inside a tile."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _data(seed, *shape, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(bf16)


@pytest.mark.parametrize("K,N,rows", [(768, 1280, (257, 1638, 3200, 3201, 6400)),   # 10 columns of 128 tiles
                                      (320, 2040, (300, 2048, 2049, 4095, 4097))])  # N ends inside a tile
def test_dense_tiles(cdx, K, N, rows):
    from complexity_deep.attention import mu_qkv_project
    from complexity_deep.linear import linear, linear_residual_
    print(f"mid tiles K={K} N={N}", flush=True)
    big = 20000
    x, w, r = _data(1, big, K), _data(2, N, K, scale=0.05), _data(3, big, N)
    mu, w2 = _data(4, big, K), _data(5, N, 2 * K, scale=0.05)
    full, added = linear(x, w), linear_residual_(x, w, r.clone())
    both = mu_qkv_project(x[None], mu[None], w2, K)[0]
    for m in rows:
        assert torch.equal(linear(x[:m].contiguous(), w), full[:m]), m
        assert torch.equal(linear_residual_(x[:m].contiguous(), w, r[:m].clone()), added[:m]), m
        assert torch.equal(mu_qkv_project(x[None, :m].contiguous(), mu[None, :m].contiguous(), w2, K)[0], both[:m]), m


@pytest.mark.parametrize("H,ie,E,shared", [(768, 512, 4, True), (1280, 864, 4, True), (512, 200, 3, False), (2048, 704, 8, True)])
def test_moe_tiles(cdx, H, ie, E, shared):
    print(f"mid tiles moe H={H} ie={ie} E={E}", flush=True)
    torch.manual_seed(H)
    m = cdx.TokenRoutedMLP(H, ie * E, num_experts=E, vocab_size=999, shared_expert=shared).to(bf16).cuda()
    big = 16384
    ids = torch.randint(0, 999, (1, big), device="cuda")
    x, r = _data(1, 1, big, H), _data(2, 1, big, H)
    with torch.no_grad():
        full, added = m(x, token_ids=ids), m(x, token_ids=ids, residual=r.clone())
        for t in (65, 700, 1000, 2048, 3001, 6000, 8192):
            a = m(x[:, :t].contiguous(), token_ids=ids[:, :t].contiguous())
            assert torch.equal(a, full[:, :t]), t
            b = m(x[:, :t].contiguous(), token_ids=ids[:, :t].contiguous(), residual=r[:, :t].clone())
            assert torch.equal(b, added[:, :t]), t


@pytest.mark.parametrize("K,N,rows", [(832, 1280, (3201, 6400, 6401, 6528, 6529)),  # K past the short products: pairs of
                                      (2048, 4096, (1400, 2048, 2049)),             # tiles from 6401 rows (26 x 5 squares)
                                      (768, 3408, (1200, 2304)), (768, 3416, (1200, 2304)), (512, 8192, (600, 1024))])
def test_dense_tiles_where_pairs_of_tiles_end(cdx, K, N, rows):
    from complexity_deep.linear import linear
    print(f"mid tiles, pairs K={K} N={N}", flush=True)
    x, w = _data(1, 16384, K), _data(2, N, K, scale=0.05)
    full = linear(x, w)
    for m in rows:
        assert torch.equal(linear(x[:m].contiguous(), w), full[:m]), m


@pytest.mark.parametrize("H,ie,E,T", [(256, 64, 64, (66, 200, 5900, 6100)), (2048, 704, 8, (777, 1000, 2500, 3900)),
                                      (512, 512, 32, (70, 400, 1700, 3000))])
def test_moe_tiles_of_many_experts(cdx, H, ie, E, T):
    """One tile per expert, segments around one tile long, and some that are empty."""
    print(f"mid tiles moe of many experts H={H} E={E}", flush=True)
    torch.manual_seed(E)
    m = cdx.TokenRoutedMLP(H, ie * E, num_experts=E, vocab_size=999).to(bf16).cuda()
    big = 32768
    ids = torch.randint(0, 999, (1, big), device="cuda")
    x = _data(1, 1, big, H)
    with torch.no_grad():
        full = m(x, token_ids=ids)
        for t in T:
            assert torch.equal(m(x[:, :t].contiguous(), token_ids=ids[:, :t].contiguous()), full[:, :t]), t


@pytest.mark.parametrize("H,nq,nkv,B,b,S", [(768, 12, 4, 40, 8, 512), (768, 12, 4, 50, 13, 333), (768, 12, 4, 40, 13, 500),
                                            (768, 12, 4, 24, 6, 777), (512, 16, 4, 64, 20, 333), (512, 16, 4, 32, 12, 512),
                                            (1280, 20, 4, 24, 6, 520)])
@pytest.mark.parametrize("vt,side", [(True, True), (True, False), (False, True)])
def test_rope_tiles(cdx, H, nq, nkv, B, b, S, vt, side):
    """mu-QKV + RoPE at heads of 64 and 32 with one to two 128 x 128 tiles per CU: the first b
    sequences alone equal the same sequences of a batch of 256 x 256 tiles, with x and mu side
    by side (one operand) and apart."""
    from complexity_deep.attention import mu_qkv_rope
    from complexity_deep.rotary import RotaryEmbedding
    D = H // nq
    print(f"mid tiles, rope H={H} D={D} b={b} S={S} vt={vt} side={side}", flush=True)
    w = _data(2, (nq + 2 * nkv) * D, 2 * H, scale=0.02)
    qn, kn = _data(3, D, scale=0.1) + 1, _data(4, D, scale=0.1) + 1
    table = RotaryEmbedding(D).cuda().cos_sin_table(S, torch.device("cuda"))
    pair = _data(1, B, S, 2 * H)

    def run(n):
        t = pair[:n]
        x, mu = t[..., :H], t[..., H:]
        if not side:
            x, mu = x.contiguous(), mu.contiguous()
        return mu_qkv_rope(x, mu, w, H, nq, nkv, D, qn, kn, 1e-6, table, 0, v_transposed=vt)

    for a, c, what in zip(run(b), run(B), "qkv"):
        if what == "v" and vt:
            a, c = a[..., :S // 16 * 16], c[..., :S // 16 * 16]
        assert torch.equal(a, c[:b]), what
