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
