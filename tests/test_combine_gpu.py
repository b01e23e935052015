"""Calls large enough for the sum's skipping loads (2 MiB of partial rows):
tokens with all, some and none of their slots routed here, at a batch of
slots' edge (16) and past it."""

from __future__ import annotations

import pytest
import torch

from test_fused_gpu import _check, _make, mfma_experts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("topk,M,K", [(10, 420, 512), (16, 300, 512), (17, 280, 512),
                                      (40, 120, 512), (15, 777, 608), (10, 400, 1056)])
def test_skipped_slots(pkg, orc, synth, dev, topk, M, K):
    """K = 608 and 1,056: rows that end inside a wave."""
    shape = synth.LayerShape(E=64, topk=topk, K=K, N=256, group=32)
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, M, dev, seed=topk)
    g = torch.Generator().manual_seed(M)
    keep = torch.rand((M, 1), generator=g) * 1.2 - 0.1  # some rows whole, some empty
    drop = torch.rand((M, topk), generator=g) > keep
    bad = torch.where(torch.rand((M, topk), generator=g) < 0.5, -1, shape.E)
    ti = torch.where(drop.to(dev), bad.to(torch.int32).to(dev), ti).contiguous()
    print(f"skipped slots topk={topk} M={M} K={K} dropped={int(drop.sum())}", flush=True)
    # a call before with every row written: skipped rows must not show through
    pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, torch.zeros_like(ti), 32)
    out = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, 32)
    torch.cuda.synchronize()
    assert bool((out[(drop.all(1)).to(dev)] == 0).all())
    _check(orc, out, x, w13, w2, s13, s2, tw, ti, 32, f"skipped slots topk={topk}",
           bf16_experts=mfma_experts(pkg, ti, shape.E, shape.N, shape.K))
