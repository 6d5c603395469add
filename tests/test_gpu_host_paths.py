"""The operators' native call paths (complexity_deep._host) against the general Python paths
they stand in for (taken while a timing hook is set): the same bits over the operand forms
both accept (contiguous, strided, broadcast, cached), and the forms that the native paths
leave to the general one (they return None and the call still works or raises)."""

from __future__ import annotations

import pytest
import torch

from _metrics import errors

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _both(fn):
    from complexity_deep import _native as nat
    with torch.no_grad():
        a = fn()
        nat.set_launch_hook(lambda *args: None)
        try:
            b = fn()
        finally:
            nat.set_launch_hook(None)
    return a, b


def _same(a, b, what):
    if isinstance(a, torch.Tensor):
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b), what
    elif isinstance(a, (tuple, list)):
        assert len(a) == len(b), what
        for x, y in zip(a, b):
            _same(x, y, what)
    elif hasattr(a, "perm"):
        _same([a.expert_id, a.perm, a.inv_perm, a.counts, a.offsets],
              [b.expert_id, b.perm, b.inv_perm, b.counts, b.offsets], what)
    else:
        assert a == b, what


def _near(a, b, what):
    """Two bf16 computations of one value that round at different places: each is off the
    exact one by bf16 roundings (2^-9 of a value, a few of them through the layers), so they
    differ by at most twice that."""
    e = errors(a, b)
    assert e["rel_rms"] <= 1e-2 and e["max_rel"] <= 2e-2, f"{what}: {e}"


def _new(*shape, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g).to(bf16).cuda()


def test_operators(cdx):
    from complexity_deep.layer import mu_guidance
    from complexity_deep.linear import embedding, linear, linear_accumulate_
    from complexity_deep.normalization import add_rms_norm, rms_norm
    print("host paths: operators", flush=True)
    x, r, w = _new(3, 7, 256), _new(3, 7, 256, seed=1), _new(256)
    ids = torch.randint(-2, 503, (3, 7), device="cuda")
    maps = [torch.randint(0, 5, (500,), device="cuda") for _ in range(2)]
    wl, wm = _new(512, 256), _new(256, 256)

    def pair(fn, half):
        buf = torch.zeros(3, 7, 512, dtype=bf16, device="cuda")
        fn(buf[..., :256] if half == 0 else buf[..., 256:])
        return buf

    cases = {
        "rms_norm": lambda: rms_norm(x, w, 1e-6),
        "rms_norm strided x": lambda: rms_norm(x.transpose(0, 1), w, 1e-6),
        "rms_norm fp32 weight": lambda: rms_norm(x, w.float(), 1e-6),
        "rms_norm out": lambda: pair(lambda o: rms_norm(x, w, 1e-6, out=o), 0),
        "rms_norm empty": lambda: rms_norm(x[:0], w, 1e-6),
        "add_rms_norm": lambda: add_rms_norm(x, r, w, 1e-6),
        "add_rms_norm no residual kept": lambda: add_rms_norm(x, r, w, 1e-6, store_residual=False),
        "add_rms_norm strided": lambda: add_rms_norm(x.transpose(0, 1), r.transpose(0, 1), w, 1e-6),
        "embedding": lambda: embedding(ids.clamp(0, 255), wm),
        "embedding int32": lambda: embedding(ids.clamp(0, 255).int(), wm),
        "linear": lambda: linear(x, wl),
        "linear ragged N": lambda: linear(x, wl[:509].contiguous()),
        "linear strided x": lambda: linear(x.transpose(0, 1), wl),
        "linear_accumulate_": lambda: linear_accumulate_(x, wm, r.clone()),
        "mu_guidance": lambda: mu_guidance(x, wm, w, 0.0, 2.0, -2.0, 2.0),
        "mu_guidance out": lambda: pair(lambda o: mu_guidance(x, wm, w, 0.0, 2.0, out=o), 1),
        "mu_guidance strided": lambda: mu_guidance(x.transpose(0, 1), wm.t(), w),
        "route_plan": lambda: cdx.route_plan(ids, maps[0], 5),
        "route_plan int32 ids": lambda: cdx.route_plan(ids.int(), maps[0], 5),
        "route_plan expert ids": lambda: cdx.route_plan(ids, None, 5),
        "route_plan empty": lambda: cdx.route_plan(ids[:0], maps[0], 5),
        "route_plans": lambda: cdx.route_plans(ids, maps, 5),
        "route_plans int32 maps": lambda: cdx.route_plans(ids, [m.int() for m in maps], 5),
    }
    for what, fn in cases.items():
        _same(*_both(fn), what)
    for bad in (lambda: rms_norm(x, w[:8], 1e-6), lambda: linear(x, wl[:, :128].contiguous()),
                lambda: mu_guidance(x, wm, w[:8]), lambda: add_rms_norm(x, r[:1], w, 1e-6),
                lambda: rms_norm(x.cpu(), w, 1e-6), lambda: rms_norm(x.half(), w, 1e-6)):
        with pytest.raises((RuntimeError, ValueError)):
            bad()


@pytest.mark.parametrize("T,H,I,E,offs", [(40, 128, 64, 3, (3, 20, 20, 37)), (700, 256, 72, 2, (0, 300, 700)),
                                          (513, 320, 200, 4, (100, 100, 256, 400, 512)), (300, 64, 8, 1, (0, 0))])
def test_expert_operators(cdx, T, H, I, E, offs):
    print(f"host paths: experts T={T} H={H} I={I} E={E}", flush=True)
    x = _new(T, H)
    gate, up, down = (_new(*s, seed=3) * 0.1 for s in ((E, H, I), (E, H, I), (E, I, H)))
    offsets = torch.tensor(offs, device="cuda")
    for what, fn in {
            "cggr": lambda: cdx.persistent_swiglu_cggr(x, gate, up, down, offsets),
            "cggr int32 offsets": lambda: cdx.persistent_swiglu_cggr(x, gate, up, down, offsets.int()),
            "cggr strided weights": lambda: cdx.persistent_swiglu_cggr(
                x, gate.transpose(1, 2).contiguous().transpose(1, 2), up, down, offsets),
            "cggr strided rows": lambda: cdx.persistent_swiglu_cggr(x.t().contiguous().t(), gate, up, down, offsets)}.items():
        _same(*_both(fn), what)
    ids = torch.randint(-1, E + 1, (T,), device="cuda")  # out of range: clamped
    for t in (x, x[:, :7].contiguous(), x.float(), x.view(T, 2, -1)):
        for i in (ids, ids.int()):
            _same(*_both(lambda: cdx.sort_tokens_by_expert(t, i, E)), f"sort {t.dtype} {tuple(t.shape)}")


@pytest.mark.parametrize("H,nq,nkv", [(256, 4, 2), (320, 8, 4), (512, 4, 4)])
def test_attention(cdx, H, nq, nkv):
    print(f"host paths: attention H={H} heads={nq}/{nkv}", flush=True)
    torch.manual_seed(H)
    m = cdx.ComplexityAttention(H, nq, nkv).to(bf16).cuda().eval()
    D = H // nq
    pair = _new(2, 150, 2 * H)
    row = _new(1, 1, H)
    for S in (1, 5, 20, 150):
        x, mu = pair[:, :S, :H], pair[:, :S, H:]  # evenly spaced rows for S = 150 only
        kv = tuple(_new(2, nkv, 33, D, seed=s) for s in (3, 4))
        for what, args in {"contiguous": (x.contiguous(), mu.contiguous()), "halves": (x, mu), "no mu": (x, None),
                           "one mu row": (x.contiguous(), row.expand(2, S, H)), "mu of [1, S, H]": (x, mu[:1]),
                           "mu per sequence": (x, mu[:, :1].expand(2, S, H))}.items():
            for past in (None, kv):
                for cache in (False, True):
                    _same(*_both(lambda: m(args[0], mu_prev=args[1], past_key_value=past, use_cache=cache)),
                          f"{what} S={S} past={past is not None} cache={cache}")


def test_moe_and_model(cdx):
    print("host paths: moe, model", flush=True)
    torch.manual_seed(2)
    moe = cdx.TokenRoutedMLP(256, 704, num_experts=4, vocab_size=500).to(bf16).cuda()
    ids = torch.randint(0, 500, (3, 50), device="cuda")
    x, r = _new(3, 50, 256), _new(3, 50, 256, seed=9)
    for what, fn in {"moe": lambda: moe(x, token_ids=ids), "residual": lambda: moe(x, token_ids=ids, residual=r.clone()),
                     "strided": lambda: moe(x.transpose(0, 1), token_ids=ids.t()), "average": lambda: moe(x)}.items():
        _same(*_both(fn), what)
    moe.up_proj_w.data.mul_(2)  # in place: seen by both
    moe.gate_proj_w = torch.nn.Parameter(moe.gate_proj_w.detach().clone())  # replaced: bound again
    _same(*_both(lambda: moe(x, token_ids=ids)), "after writes")
    cfg = cdx.ComplexityConfig(vocab_size=500, hidden_size=256, intermediate_size=704, num_hidden_layers=3,
                               num_attention_heads=4, num_key_value_heads=2, num_experts=4)
    model = cdx.ComplexityModel(cfg).to(bf16).cuda().eval()
    _same(*_both(lambda: model(ids).logits), "model")
    # (A step of at most 8 rows folds its norms into the products on the native path only.)
    _near(*_both(lambda: model(ids[:, :1]).logits), "model, one token")
    with torch.no_grad():
        past = model(ids, use_cache=True).past_key_values
    a, b = _both(lambda: model(ids[:, -1:], past_key_values=past, use_cache=True))
    _near(a.logits, b.logits, "step")
    for x, y in zip([t for kv in a.past_key_values for t in kv], [t for kv in b.past_key_values for t in kv]):
        _near(x, y, "step cache")


@pytest.mark.parametrize("H,I,nq,nkv,E,B,S,past", [(256, 704, 4, 2, 4, 1, 1, 9), (320, 896, 8, 4, 4, 2, 4, 30),
                                                   (512, 1408, 4, 4, 8, 8, 1, 5), (1280, 3456, 16, 4, 4, 1, 3, 0)])
def test_block_step(cdx, oracle, H, I, nq, nkv, E, B, S, past):
    """A step's block with folded norms against the block's separate norms, with large and small
    hidden states (the folded product scales after the sum)."""
    from complexity_deep.normalization import rms_norm
    print(f"block step H={H} B={B} S={S} past={past}", flush=True)
    torch.manual_seed(H)
    blk = cdx.TransformerBlock(H, I, nq, nkv, num_experts=E, vocab_size=500).to(bf16).cuda().eval()
    with torch.no_grad():
        for n, p in blk.named_parameters():
            if "norm" in n:
                p.normal_(1, 0.2)
        blk.mu_guidance.mu_proj.weight.normal_(0, 0.02)
    D = H // nq
    ids = torch.randint(0, 500, (B, S), device="cuda")
    kv = (_new(B, nkv, past, D), _new(B, nkv, past, D, seed=1)) if past else None
    mu = _new(B, S, H, seed=5)
    nxt = cdx.RMSNorm(H).to(bf16).cuda()
    for scale in (1.0, 64.0, 2.0 ** -6):
        h = _new(B, S, H) * scale
        with torch.no_grad():
            plan = blk.mlp.plan(ids)
            a = h.clone()
            (k, v), mu_a = blk.step(a, mu, kv, plan)
            b = h.clone()
            normed = rms_norm(b, blk.input_layernorm.weight, 1e-6)
            _, _, kv_b, mu_b = blk.forward_fused(b, normed, nxt, past_key_value=kv, use_cache=True, token_ids=ids,
                                                 mu_prev=mu, route=plan)
        for x, y, what in ((a, b, "h"), (k, kv_b[0], "k"), (v, kv_b[1], "v"), (mu_a, mu_b, "mu")):
            _near(x, y, f"{what}, scale {scale}")
    blk.self_attn.register_forward_hook(lambda *a: None)
    assert blk.step(h.clone(), mu, kv, plan) is None  # a hook is not passed by


@pytest.mark.parametrize("H,nq,nkv", [(256, 4, 2), (320, 8, 4)])
def test_one_mu_row_for_every_token_takes_the_native_paths(cdx, H, nq, nkv):
    """mu of [1, 1, H] expanded to the batch (a model's first layer) is one broadcast row
    whatever the sizes are: expand() keeps the old stride in dimensions of size 1."""
    from complexity_deep import _native as nat
    print(f"host paths: one mu row, H={H}", flush=True)
    torch.manual_seed(H)
    blk = cdx.TransformerBlock(H, 704, nq, nkv, num_experts=4, vocab_size=500).to(bf16).cuda().eval()
    m, row = blk.self_attn, _new(1, 1, H)
    norms = (m.q_norm.weight, m.k_norm.weight, m.q_norm.eps)
    for B, S in ((4, 1), (1, 4), (2, 3), (1, 150), (3, 50)):
        x, mu = _new(B, S, H), row.expand(B, S, H)
        with torch.no_grad():
            table = m.rotary_emb.cos_sin_table(S, x.device)
            assert nat.host().attention(x, mu, m._qkv_w.buffer(m), nq, nkv, H // nq, *norms, table, None, None,
                                        True if B * S <= 8 else False) is not None, (B, S)
            if B * S <= 8:
                plan = blk.mlp.plan(torch.zeros(B, S, dtype=torch.long, device="cuda"))
                assert blk.step(x.clone(), mu, None, plan) is not None, (B, S)
            a, b = _both(lambda: m(x, mu_prev=mu)[0])
            c = m(x, mu_prev=mu.contiguous())[0]
        _same(a, b, (B, S))
        _near(a, c, (B, S))


def test_linear_accumulate_checks_every_size(cdx):
    """A weight without rows, and a residual of the right row count but other leading sizes, raise
    on both paths."""
    from complexity_deep import _native as nat
    from complexity_deep.linear import linear_accumulate_
    print("host paths: linear_accumulate_ sizes", flush=True)
    x, w = _new(2, 3, 128), _new(64, 128)
    for res, weight in ((_new(2, 3, 64)[..., :0], w[:0]), (_new(6, 64), w), (_new(2, 64), w), (_new(2, 3, 56), w)):
        for hook in (None, lambda *a: None):
            nat.set_launch_hook(hook)
            try:
                with pytest.raises((ValueError, RuntimeError)), torch.no_grad():
                    linear_accumulate_(x, weight, res)
            finally:
                nat.set_launch_hook(None)


@pytest.mark.parametrize("B,S,past", [(2, 1, 4), (1, 7, 7), (1, 8, 0)])
def test_block_step_of_a_wide_projection(cdx, B, S, past):
    """9216 columns of q, k and v (3072 wide, as many KV heads as query heads): the folded norm on
    the blocks of 32 output columns, which the narrower projections of test_block_step do not take."""
    from complexity_deep.normalization import rms_norm
    print(f"block step, wide projection B={B} S={S} past={past}", flush=True)
    H, heads, D = 3072, 24, 128
    torch.manual_seed(S)
    blk = cdx.TransformerBlock(H, 1024, heads, heads, num_experts=2, vocab_size=500,
                               use_mu_guidance=False).to(bf16).cuda().eval()
    with torch.no_grad():
        blk.input_layernorm.weight.normal_(1, 0.2)
    ids = torch.randint(0, 500, (B, S), device="cuda")
    kv = (_new(B, heads, past, D), _new(B, heads, past, D, seed=1)) if past else None
    mu, h = _new(B, S, H, seed=5), _new(B, S, H)
    nxt = cdx.RMSNorm(H).to(bf16).cuda()
    with torch.no_grad():
        plan = blk.mlp.plan(ids)
        a, b = h.clone(), h.clone()
        (k, v), none = blk.step(a, mu, kv, plan)
        _, _, kv_b, _ = blk.forward_fused(b, rms_norm(b, blk.input_layernorm.weight, 1e-6), nxt, past_key_value=kv,
                                          use_cache=True, token_ids=ids, mu_prev=mu, route=plan)
    assert none is None
    for x, y, what in ((a, b, "h"), (k, kv_b[0], "k"), (v, kv_b[1], "v")):
        _near(x, y, what)
