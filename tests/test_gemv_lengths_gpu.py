"""GEMV row lengths known only at run time: every remainder of the step ring and
of the staged pieces, against the oracle, and the one-launch w2 + sum of every
unrolled length (and past them) against the separate kernels; and the GEMV over
the sorted blocks, of calls with fewer than two pairs per expert that do not
route themselves."""

from __future__ import annotations

import pytest
import torch

from test_fused_gpu import _check, _make

pytestmark = pytest.mark.gpu


# Steps of 256 elements: K from one partial step to 17 (more than two staged
# pieces of 256 octets), N from one to nine.
@pytest.mark.parametrize("K,N", [(32, 32), (288, 224), (512, 544), (1056, 768), (1280, 992),
                                 (2048, 1312), (2080, 1568), (2304, 1824), (4128, 2080),
                                 (4352, 2304)])
@pytest.mark.parametrize("M", [3, 7, 14])
def test_run_time_lengths(pkg, orc, synth, dev, K, N, M):
    tag = f"lengths K={K} N={N} M={M}"
    print(tag, flush=True)
    shape = synth.LayerShape(E=6, topk=3, K=K, N=N, group=32)
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, M, dev, seed=K + M)
    out = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, 32)
    if M <= 4:
        split = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, 32,
                                        tuning=pkg.Tuning(w2_fused_max_m=1))
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), split.view(torch.int16)), tag
    torch.cuda.synchronize()
    # A flipped bf16 intermediate moves an output by its weight (up to 1 / 3 and
    # more) times its ulp: the bound of test_fused_sweep_gpu.py, ~2e-3 of
    # max|out| at a weight of one; few rows, so a flip shows in many of them.
    _check(orc, out, x, w13, w2, s13, s2, tw, ti, 32, tag, mismatch_max=0.05, excess_max=2e-3)


@pytest.mark.parametrize("K,N,group", [(1536, 320, 32), (3072, 96, 32), (1024, 448, 64),
                                       (1280, 384, 128)])
@pytest.mark.parametrize("M", [25, 47])
@pytest.mark.parametrize("form", ["uniform", "hot", "dropped"])
def test_sorted_blocks(pkg, orc, synth, dev, K, N, group, M, form):
    """hot: one expert in every token (several 16-slot blocks); dropped: ids
    outside the layer among the others."""
    tag = f"sorted K={K} N={N} G={group} M={M} {form}"
    print(tag, flush=True)
    L = pkg._lib
    shape = synth.LayerShape(E=128, topk=4, K=K, N=N, group=group)
    off = L.workspace_layout(M, 4, 128, N, K, group)
    assert L.stage_launches(M, 4, 128, N, K, group, None) == [1, 1, 1, 1]
    assert off[L.WS_GEMV_BLOCKS] - off[L.WS_TILES] == 256  # no tiles
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, M, dev, seed=K + M)
    if form == "hot":
        ti[:, 2] = 7
    elif form == "dropped":
        ti[::3, 1] = -1
        ti[1::3, 3] = 128
    out = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, group)
    torch.cuda.synchronize()
    _check(orc, out, x, w13, w2, s13, s2, tw, ti, group, tag, mismatch_max=0.05, excess_max=2e-3)
