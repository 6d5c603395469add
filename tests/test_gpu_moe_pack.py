"""cdx_moe_pack (expert weights [in, out] into the MoE kernels' operands) against strided
tensor copies, bit for bit, with widths that end inside a tile and padded units."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


@pytest.mark.parametrize("E,H,I", [(1, 64, 8), (4, 768, 512), (3, 320, 224), (2, 128, 72), (5, 2048, 56)])
def test_pack_equals_strided_copies(cdx, E, H, I):
    from complexity_deep.token_routed_mlp import pack_moe_weights
    print(f"moe pack E={E} H={H} I={I}", flush=True)
    gate, up, down = (torch.randn(*s, device="cuda").to(bf16) for s in ((E, H, I), (E, H, I), (E, I, H)))
    got = pack_moe_weights(gate, up, down, None, None, None)
    # Strided weights (the same values) take the copies.
    apart = [w.transpose(1, 2).contiguous().transpose(1, 2) for w in (gate, up, down)]
    ref = pack_moe_weights(*apart, None, None, None)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
