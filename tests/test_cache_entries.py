"""A cache entry that carries more than (k, v) is read by index, as core/attention.py:157-161
reads it."""

import types

import pytest
import torch

import complexity_deep.layer as layer_mod
from complexity_deep import _native as nat


def test_step_and_cache_check_read_the_first_two_of_an_entry(monkeypatch):
    seen = []
    monkeypatch.setattr(nat, "host", lambda: types.SimpleNamespace(block_step=lambda *a: seen.append(a[12:14])))
    block = layer_mod.TransformerBlock(64, 128, 2, 1, num_experts=2, vocab_size=32).bfloat16()
    k, v = torch.zeros(2, 1, 1, 3, 32, dtype=torch.bfloat16)
    h = torch.zeros(1, 1, 64, dtype=torch.bfloat16)
    entry = (k, v, "more")
    block.step(h, None, entry, types.SimpleNamespace(perm=None, offsets=None, num_experts=2))
    assert seen[0][0] is k and seen[0][1] is v
    assert block.self_attn._cache_fits(entry, h)


def test_general_path_reads_a_stacked_entry(monkeypatch):
    """One [2, B, heads, rows, D] tensor in the place of (k, v): its truth value is never taken."""
    from complexity_deep import attention
    seen = []

    class Stop(Exception):
        pass

    def require(*tensors, **_):
        seen.extend(tensors)
        raise Stop

    monkeypatch.setattr(nat, "require_device", require)
    x, w = torch.zeros(1, 1, 64, dtype=torch.bfloat16), torch.zeros(128, 128, dtype=torch.bfloat16)
    past = torch.zeros(2, 1, 1, 3, 32, dtype=torch.bfloat16)
    with pytest.raises(Stop):
        attention.qkv_cache(x, None, w[:, :64], w[:, 64:], 64, 2, 1, 32, None, None, 0.0, torch.zeros(4, 16, 2), past)
    assert [t.data_ptr() for t in seen[-2:]] == [past[0].data_ptr(), past[1].data_ptr()]


def test_calls_past_the_kernels_counts_keep_the_torch_path():
    """cdx_qkv_cache_fwd counts the cache's 16-byte pieces, and (token, head) rows, in 31 bits:
    a prompt beyond that, with or without a cache, is not given to it."""
    from complexity_deep.attention import ComplexityAttention
    with torch.device("meta"):
        attn = ComplexityAttention(320, 8, 4).bfloat16()
        few_kv = ComplexityAttention(1024, 128, 1).bfloat16()

    def fits(m, tokens, past=None):
        return m._cache_fits(past, torch.empty(1, tokens, m.hidden_size, dtype=torch.bfloat16, device="meta"))

    edge = 2 ** 31 // (2 * 4 * 5)  # 2 x 4 KV heads of 40, five pieces each
    assert fits(attn, edge) and not fits(attn, edge + 1)
    rows = 2 ** 31 // 130
    assert fits(few_kv, rows) and not fits(few_kv, rows + 1)
