"""Calls laid out for the exact-weight tiles (two or more pairs per expert by the
host's count) most of whose pairs belong to experts elsewhere: the launches run
the GEMV's items, by the counts that the sort left in the header, and give the
GEMV's bits; with more pairs they run the tiles."""

from __future__ import annotations

import pytest
import torch

from test_fused_gpu import _check

pytestmark = pytest.mark.gpu

OVER = 2048  # header[5] from here on: an expert with more than 8 pairs


def _call(synth, dev, counts, E, K, N, group, seed, topk=4, least=26):
    """Expert e < len(counts) holds counts[e] pairs; dropped pairs (-1 or past
    the last expert) bring the call to 2 E pairs and `least` tokens."""
    g = torch.Generator().manual_seed(seed)
    live = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))
    M = max(least, -(-max(2 * E, live.numel()) // topk))
    flat = torch.where(torch.rand(M * topk, generator=g) < 0.5, -1, E + 9000)
    flat[: live.numel()] = live
    ti = flat[torch.randperm(M * topk, generator=g)].reshape(M, topk).to(torch.int32).to(dev)
    tw = torch.softmax(torch.randn((M, topk), generator=g), dim=-1).to(dev)
    shape = synth.LayerShape(E=E, topk=topk, K=K, N=N, group=group)
    return (synth.make_hidden(M, K, dev, seed=seed), *synth.make_weights(shape, dev, seed=seed),
            tw, ti)


def _run(pkg, args, group):
    """(out, live rows of the intermediate, header) of one call."""
    x, w13, w2, s13, s2, tw, ti = args
    out = pkg.fused_experts_w4a16(*args, group)
    ws, off = pkg.workspace_tensor(x, ti, w13, w2, group)
    L = pkg._lib
    N = w13.shape[1] // 2
    inter = ws[off[L.WS_INTER]: off[L.WS_INTER] + ti.numel() * N * 2].view(torch.int16)
    flat = ti.reshape(-1)
    live = (flat >= 0) & (flat < w13.shape[0])
    header = ws[off[L.WS_HEADER]: off[L.WS_HEADER] + 24].view(torch.int32)
    torch.cuda.synchronize()
    return out, inter.view(-1, N)[live].clone(), header.tolist()


def _gemv(pkg, args, group):
    """The same call with so many more (unused) experts that the host lays it
    out for the GEMV over the sorted blocks."""
    x, w13, w2, s13, s2, tw, ti = args
    E, pairs = w13.shape[0], ti.numel()
    more = pairs // 2 + 1 - E

    def pad(t):
        return torch.cat([t, torch.zeros((more, *t.shape[1:]), dtype=t.dtype, device=t.device)])

    return _run(pkg, (x, pad(w13), pad(w2), pad(s13), pad(s2), tw,
                      torch.where((ti < 0) | (ti >= E), -1, ti)), group)


# One row chunk and a ragged last slab, one step and more than the ring holds,
# rows of both geometries' scale loads, and rows too long for four-row passes.
@pytest.mark.parametrize("K,N,group", [(96, 32, 32), (1056, 288, 32), (3072, 320, 64),
                                       (2048, 384, 128), (7456, 288, 32)])
@pytest.mark.parametrize("counts", [[1, 2, 0, 3, 4, 1, 0, 0], [4] * 6 + [0, 0], [0] * 8])
def test_few_pairs_give_the_gemvs_bits(pkg, orc, synth, dev, K, N, group, counts):
    tag = f"few pairs K={K} N={N} G={group} {counts}"
    print(tag, flush=True)
    args = _call(synth, dev, counts, len(counts), K, N, group, K + N)
    out, inter, header = _run(pkg, args, group)
    assert header[2] == sum(c > 0 for c in counts) and header[3] == 0
    assert header[4:] == [sum((0, 2, 2, 3, 3)[c] for c in counts), 0]
    want, want_inter, _ = _gemv(pkg, args, group)
    assert torch.equal(inter, want_inter), tag
    if N > 256:  # (w2 of shorter rows has few enough items to run its tiles)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), tag
    x, w13, w2, s13, s2, tw, ti = args
    if sum(counts):
        _check(orc, out, x, w13, w2, s13, s2, tw, ti, group, tag, mismatch_max=0.05,
               excess_max=4e-3)
    else:
        assert not out.any()


@pytest.mark.parametrize("counts,gemv", [([8, 1, 5, 0], True), ([9, 1, 5, 0], False),
                                         ([8] * 250, False), ([1] * 250, True)])
def test_the_line(pkg, orc, synth, dev, counts, gemv):
    """w13 on either side of the rule: two passes, three, and by throughput."""
    K, N, group = 512, 160, 32
    print(f"few pairs line {counts[:4]} x {len(counts)}", flush=True)
    args = _call(synth, dev, counts, len(counts), K, N, group, 7, topk=8)
    out, inter, header = _run(pkg, args, group)
    over = sum(OVER if c > 8 else c > 4 for c in counts)
    assert header[2] == sum(c > 0 for c in counts) and header[5] == over
    assert torch.equal(inter, _gemv(pkg, args, group)[1]) == gemv
    x, w13, w2, s13, s2, tw, ti = args
    _check(orc, out, x, w13, w2, s13, s2, tw, ti, group, f"line {counts[:4]}", mismatch_max=0.05,
           excess_max=4e-3)


@pytest.mark.parametrize("counts", [[1, 2, 0, 3, 4, 1, 0, 0], [1, 12, 0, 3, 70, 1, 0, 0]])
def test_after_the_many_workgroup_sort(pkg, orc, synth, dev, counts):
    """8,800 pairs, nearly all of them dropped: the sort over many workgroups
    leaves the same counts."""
    K, N = 512, 288
    print(f"few pairs, many workgroups {counts}", flush=True)
    args = _call(synth, dev, counts, len(counts), K, N, 32, 9, topk=8, least=1100)
    x, w13, w2, s13, s2, tw, ti = args
    assert pkg._lib.stage_launches(1100, 8, 8, N, K, 32, None)[0] == 2
    out, _, header = _run(pkg, args, 32)
    assert header[4:] == [sum((0, 2, 2, 3, 3)[c] if c < 5 else 6 for c in counts),
                          sum(OVER if c > 8 else c > 4 for c in counts)]
    assert header[1] == 8800 - sum(counts) and header[3] == 0
    _check(orc, out, x, w13, w2, s13, s2, tw, ti, 32, f"many workgroups {counts}",
           mismatch_max=0.05, excess_max=4e-3)


def test_one_share_of_the_experts(pkg, synth, dev):
    """32 of 256 experts and an eighth of their intermediate size, 25 tokens:
    about one pair per expert is left of the ten that the host counts."""
    E, K, N = 32, 3072, 128
    shape = synth.LayerShape(E=E, topk=10, K=K, N=N, group=32)
    w = synth.make_weights(shape, dev, seed=2)
    x = synth.make_hidden(25, K, dev, seed=2)
    tw, ti = synth.make_routing(25, 256, 10, dev, seed=2)
    args = (x, *w, tw, ti)
    out, inter, header = _run(pkg, args, 32)
    assert header[2] > 0 and header[5] < OVER
    assert torch.equal(inter, _gemv(pkg, args, 32)[1])
