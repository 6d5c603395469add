"""Routing plans of one block (up to 4096 tokens) at the edges of its chunks of 64, waves and
rounds of 1024, and just past them, bit-exact against the C oracle; several maps at once."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E", [(63, 64), (64, 1), (65, 3), (1000, 64), (2049, 8), (4095, 7), (4096, 64), (4097, 8)])
def test_plans_of_one_block(cdx, oracle, T, E):
    print(f"one-block plan T={T} E={E}", flush=True)
    rng = np.random.default_rng(T)
    ids = rng.integers(-3, 503, size=T).astype(np.int64)
    maps = [rng.integers(0, E, size=500).astype(np.int64) for _ in range(3)]
    plans = cdx.route_plans(torch.from_numpy(ids).cuda(), [torch.from_numpy(m).cuda() for m in maps], E)
    for plan, m in zip(plans, maps):
        ref = oracle.route_plan(ids, m, E)
        for k in ("expert_id", "perm", "inv_perm", "counts", "offsets"):
            np.testing.assert_array_equal(getattr(plan, k).cpu().numpy().astype(np.int64), ref[k].astype(np.int64), err_msg=k)
