"""The exact-weight MFMA tiles (csrc/xtile.hip) against the CPU oracle, at the
edges of their tiles, row tiles, steps and scale windows.

The calls are the ones that reach them: N or K no multiple of 256, scales that
are not 16-byte aligned, or a tuning that keeps every expert on exact weights,
with too many pairs to route themselves and at least two per expert; each has
an expert of more than eight pairs, without which a launch may run the GEMV's
items.  The header says that tiles were made, and of which height.  No weight
is rounded, so the bars are the tight ones of test_fused_gpu.py for exact experts.
"""

from __future__ import annotations

import pytest
import torch

from test_fused_gpu import _check, _make

pytestmark = pytest.mark.gpu

# pairs per expert: around every block of 16 slots and every tile height
COUNTS = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 97, 128, 129, 0, 200]


def _case(synth, dev, counts, K, N, group, topk, seed):
    """One call whose experts hold exactly `counts` pairs, in mixed order."""
    g = torch.Generator().manual_seed(seed)
    flat = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))
    flat = flat[torch.randperm(flat.numel(), generator=g)]
    M = flat.numel() // topk
    shape = synth.LayerShape(E=len(counts), topk=topk, K=K, N=N, group=group)
    w13, w2, s13, s2 = synth.make_weights(shape, dev, seed=seed)
    x = synth.make_hidden(M, K, dev, seed=seed)
    ti = flat[: M * topk].reshape(M, topk).to(torch.int32).to(dev)
    tw = torch.softmax(torch.randn((M, topk), generator=g), dim=-1).to(dev)
    return w13, w2, s13, s2, x, tw, ti


# The same below 24 pairs per expert on average: tiles of 32 slots.
SHORT = [1, 15, 16, 17, 31, 32, 33, 0, 70, 1, 2, 5, 9, 17, 8, 4, 3]


def _tiles_ran(pkg, x, ti, w13, w2, group, tile_m, tuning=None):
    """The last call's launches ran its tiles, of at most tile_m slots each."""
    L = pkg._lib
    ws, off = pkg.workspace_tensor(x, ti, w13, w2, group, tuning=tuning)
    h = ws[off[L.WS_HEADER]: off[L.WS_HEADER] + 24].view(torch.int32).tolist()
    E = w13.shape[0]
    flat = ti.reshape(-1).long().cpu()
    counts = torch.bincount(flat[(flat >= 0) & (flat < E)], minlength=E).tolist()
    assert h[5] >= 2048, "no expert of more than eight pairs"
    assert h[2] == sum(-(-c // tile_m) for c in counts)


# K, N, group: one 32-element chunk, partial steps and odd step counts, single
# scales (rows of no whole 16 bytes), scale windows that end inside a row, one
# row tile and several with an idle tail
SHAPES = [(32, 32, 32), (96, 160, 32), (128, 128, 32), (384, 288, 32), (1056, 704, 32),
          (2304, 512, 32), (64, 64, 64), (576, 320, 64), (2560, 1088, 64), (128, 128, 128),
          (1408, 384, 128), (2048, 1024, 128)]


@pytest.mark.parametrize("K,N,group", SHAPES)
@pytest.mark.parametrize("counts,topk", [(COUNTS, 1), ([3, 1, 0, 40, 2, 9, 1, 64, 5, 195], 4)])
def test_tiles_match_oracle(pkg, orc, synth, dev, K, N, group, counts, topk):
    tag = f"xtile K={K} N={N} G={group} topk={topk}"
    print(tag, flush=True)
    w13, w2, s13, s2, x, tw, ti = _case(synth, dev, counts, K, N, group, topk, K + N + topk)
    t = pkg.Tuning(gemv_only_max_m=pkg.tuning.ALWAYS)
    out = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, group, tuning=t)
    again = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, group, tuning=t)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))
    _tiles_ran(pkg, x, ti, w13, w2, group, 48 if group == 128 else 64, t)
    # A flipped bf16 intermediate moves an output by its weight times the
    # intermediate's ulp: with topk = 1 (weight 1) up to ~2e-3 of max|out|
    # (the bound test_fused_sweep_gpu.py derives per case), at topk = 4 a
    # quarter of that; short reductions (N <= 128 terms) leave max|out| small
    # against one term, hence twice the bound.
    _check(orc, out, x, w13, w2, s13, s2, tw, ti, group, tag, mismatch_max=0.05,
           excess_max=4e-3)


@pytest.mark.parametrize("K,N,group", SHAPES)
@pytest.mark.parametrize("topk,dropped", [(1, 0), (4, 100)])
def test_short_tiles_match_oracle(pkg, orc, synth, dev, K, N, group, topk, dropped):
    tag = f"short xtile K={K} N={N} G={group} topk={topk} dropped={dropped}"
    print(tag, flush=True)
    E = len(SHORT)
    counts = SHORT + [dropped] if dropped else SHORT
    assert sum(counts) < 24 * E
    w13, w2, s13, s2, x, tw, ti = _case(synth, dev, counts, K, N, group, topk, K + N + topk)
    w13, w2, s13, s2 = (t[:E].contiguous() for t in (w13, w2, s13, s2))
    t = pkg.Tuning(gemv_only_max_m=pkg.tuning.ALWAYS)
    out = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, group, tuning=t)
    torch.cuda.synchronize()
    _tiles_ran(pkg, x, ti, w13, w2, group, 32, t)
    _check(orc, out, x, w13, w2, s13, s2, tw, ti, group, tag, mismatch_max=0.05,
           excess_max=4e-3)


@pytest.mark.parametrize("K,N,group", [(512, 256, 32), (512, 512, 64), (1024, 1024, 128)])
def test_unaligned_scales_and_fp32_partials(pkg, orc, synth, dev, K, N, group):
    """Scales two bytes off their alignment give the aligned scales' bits, and
    four tokens with 80 slots each keep fp32 partial rows."""
    shape = synth.LayerShape(E=8, topk=80, K=K, N=N, group=group)
    w13, w2, s13, s2 = synth.make_weights(shape, dev, seed=K)
    M = 4
    x = synth.make_hidden(M, K, dev, seed=K)
    g = torch.Generator().manual_seed(K)
    ti = torch.randint(0, 8, (M, 80), generator=g).to(torch.int32).to(dev)
    tw = torch.full((M, 80), 1 / 80, device=dev)

    def shifted(s):
        buf = torch.zeros(s.numel() + 8, dtype=s.dtype, device=dev)
        buf[1: 1 + s.numel()] = s.reshape(-1)
        return buf[1: 1 + s.numel()].view(s.shape)

    print(f"xtile unaligned K={K} N={N} G={group}", flush=True)
    t = pkg.Tuning(gemv_only_max_m=pkg.tuning.ALWAYS)
    out = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, group, tuning=t)
    off = pkg.fused_experts_w4a16(x, w13, w2, shifted(s13), shifted(s2), tw, ti, group)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), off.view(torch.int16))
    _tiles_ran(pkg, x, ti, w13, w2, group, 48 if group == 128 else 64)
    _check(orc, out, x, w13, w2, s13, s2, tw, ti, group, f"unaligned G={group}",
           mismatch_max=0.05)


@pytest.mark.parametrize("K,N,group,M", [(1056, 704, 32, 120), (512, 128, 64, 300)])
def test_graph_replay(pkg, synth, dev, K, N, group, M):
    shape = synth.LayerShape(E=10, topk=3, K=K, N=N, group=group)
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, M, dev, seed=M)
    args = (w13, w2, s13, s2, tw, ti, group)
    eager = pkg.fused_experts_w4a16(x, *args)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = pkg.fused_experts_w4a16(x, *args)
    for i in range(3):
        out.zero_()
        pkg.fused_experts_w4a16(synth.make_hidden(M, K, dev, seed=70 + i), *args)
        torch.cuda.synchronize()
        print(f"xtile replay {i} K={K} N={N}", flush=True)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16)), f"replay {i}"
    del g
    pkg.release_graph_workspaces()
