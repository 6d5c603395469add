"""mu-QKV + RoPE at head dim 128 on 128-column tiles (few tokens: 128-row tiles, then 256-row
ones) against the 256 x 256 tiles of a larger batch: the first sequences alone and inside the
batch give the same bits, with sequences that end inside a tile and with both V layouts."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


@pytest.mark.parametrize("b,B,S,vt,norm", [(1, 40, 129, True, True), (1, 40, 128, True, True), (3, 24, 333, False, True),
                                           (4, 32, 256, True, False), (3, 16, 500, True, True), (1, 9, 1100, True, True)])
def test_head_tiles_equal_square_tiles(cdx, b, B, S, vt, norm):
    from complexity_deep.attention import mu_qkv_rope
    from complexity_deep.rotary import RotaryEmbedding
    H, nq, nkv, D = 1024, 8, 4, 128
    print(f"head tiles b={b} B={B} S={S} vt={vt} norm={norm}", flush=True)
    g = torch.Generator().manual_seed(S)
    x = torch.randn(B, S, H, generator=g).to(bf16).cuda()
    mu = torch.randn(B, S, H, generator=g).to(bf16).cuda()
    w = (torch.randn((nq + 2 * nkv) * D, 2 * H, generator=g) * 0.02).to(bf16).cuda()
    qn = (1 + 0.1 * torch.randn(D, generator=g)).to(bf16).cuda() if norm else None
    table = RotaryEmbedding(D).cuda().cos_sin_table(S, torch.device("cuda"))
    full = mu_qkv_rope(x, mu, w, H, nq, nkv, D, qn, qn, 1e-6, table, 0, v_transposed=vt)
    part = mu_qkv_rope(x[:b].contiguous(), mu[:b].contiguous(), w, H, nq, nkv, D, qn, qn, 1e-6, table, 0,
                       v_transposed=vt)
    for a, c, what in zip(part, full, "qkv"):
        if what == "v" and vt:
            a, c = a[..., :S // 16 * 16], c[..., :S // 16 * 16]
        assert torch.equal(a, c[:b]), what
