"""The native call path (csrc/fastcall.cpp): the calls it takes give the Python
path's bits, and it leaves every other call to that path."""

from __future__ import annotations

import threading

import pytest
import torch

from test_fused_gpu import _make


@pytest.fixture(autouse=True)
def no_tuning_variables(monkeypatch):
    """The native path takes no calls while they are set (conftest.py does)."""
    for var in ("W4A16_MOE_TUNING", "W4A16_MOE_CONFIG_DIR"):
        monkeypatch.delenv(var, raising=False)


def test_host_tensors_are_left_alone(pkg):
    f = pkg._lib.fast()
    t = torch.zeros(2, 2)
    assert f.fused(t, t, t, t, t, t, t, 32) is None
    assert f.router(t, 1, True) is None
    assert f.align(t, 16, 4) is None
    with pytest.raises(pkg._lib.W4A16Error):
        pkg.fused_experts_w4a16(t, t, t, t, t, t, t)


@pytest.fixture(params=["missing", "not loadable"])
def no_native_module(request, pkg, monkeypatch, tmp_path):
    """The module cannot be loaded; gives the loaded one."""
    native = pkg._lib.load_fast()
    path = tmp_path / "w4a16_fastcall.so"
    if request.param == "not loadable":
        path.write_bytes(b"not a library")
    monkeypatch.setattr(pkg._lib, "FAST_PATH", path)
    monkeypatch.setattr(pkg._lib, "_fast", None)
    yield native
    pkg.w4a16_moe._WS_POOL.clear()  # the next buffers are shown to the module again


def test_without_the_native_module(pkg, no_native_module, monkeypatch):
    """The path in Python needs the HIP library only: arguments are checked as
    ever, and with no library at all too; the pool can be cleared."""
    pkg.w4a16_moe._WS_POOL.clear()
    t = torch.zeros(2, 2)
    with pytest.raises(ImportError):
        pkg._lib.load_fast()
    calls = [lambda: pkg.fused_experts_w4a16(t, t, t, t, t, t, t),
             lambda: pkg.moe_align_block_size(t, 16, 4), lambda: pkg.router_topk_softmax(t, 1)]
    with pytest.warns(RuntimeWarning, match="native call path"):
        pkg._lib.fast()
    with pytest.raises(ImportError):  # (still, with the stand-in in its place)
        pkg._lib.load_fast()
    for has_library in (True, False):
        if not has_library:
            monkeypatch.setattr(pkg._lib, "LIB_PATH", pkg._lib.FAST_PATH.parent / "none.so")
            monkeypatch.setattr(pkg._lib, "_fast", None)
        for call in calls:
            with pytest.raises(pkg._lib.W4A16Error):
                call()


SHAPES = [(16, 4, 512, 256, 32, 6), (16, 4, 512, 256, 64, 40), (8, 2, 96, 160, 32, 90),
          (256, 10, 3072, 1024, 32, 1)]


def _bits(t):
    return t.view(torch.int16)


@pytest.mark.gpu
@pytest.mark.parametrize("E,topk,K,N,group,M", SHAPES)
def test_same_bits_as_the_python_path(pkg, synth, dev, monkeypatch, E, topk, K, N, group, M):
    shape = synth.LayerShape(E=E, topk=topk, K=K, N=N, group=group)
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, M, dev, seed=M)
    f = pkg._lib.fast()
    f.clear_plans()
    args = (x, w13, w2, s13, s2, tw, ti, group)
    assert f.fused(*args) is None  # no plan yet
    first = pkg.fused_experts_w4a16(*args)
    fast = f.fused(*args)
    assert isinstance(fast, torch.Tensor) and fast.shape == first.shape
    assert torch.equal(_bits(fast), _bits(first))
    wide = torch.zeros(M, K + 64, dtype=torch.bfloat16, device=dev)
    wide[:, 32: 32 + K] = x
    forms = [(wide[:, 32: 32 + K], w13.view(torch.uint8), w2.view(torch.uint8), s13, s2, tw,
              ti.to(torch.int64), group),
             (x, w13, w2, s13, s2, tw.t().contiguous().t(), ti.t().contiguous().t(), group)]
    for a in forms:
        assert torch.equal(_bits(f.fused(*a)), _bits(first))
    # calls of a form or a moment it does not know
    odd = torch.zeros(M, K + 4, dtype=torch.bfloat16, device=dev)[:, :K]  # row stride
    assert f.fused(odd, *args[1:]) is None or odd.stride(0) % 8 == 0
    assert f.fused(x.float(), *args[1:]) is None
    assert f.fused(x, w13, w2, s13[:, ::2], s2, tw, ti, group) is None
    assert f.fused(x, w13, w2, s13, s2, tw[:, :1], ti, group) is None
    assert f.fused(x[:0], w13, w2, s13, s2, tw[:0], ti[:0], group) is None
    assert f.fused(x.as_subclass(type("Sub", (torch.Tensor,), {})), *args[1:]) is None
    for var in ("W4A16_MOE_TUNING", "W4A16_MOE_CONFIG_DIR"):
        monkeypatch.setenv(var, "default")
        assert f.fused(*args) is None
        monkeypatch.delenv(var)
    with pytest.raises(pkg._lib.W4A16Error):
        pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw[:, :1], ti, group)
    with torch.device("cuda:0"):  # a torch-function mode
        assert f.fused(*args) is None


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:the native call path")
def test_same_bits_without_the_native_module(pkg, synth, dev, no_native_module, monkeypatch):
    shape = synth.LayerShape(E=16, topk=4, K=512, N=256, group=32)
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, 6, dev, seed=6)
    logits = torch.randn((6, 16), device=dev)

    def calls():
        return [pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, 32),
                *pkg.router_topk_softmax(logits, 4), *pkg.moe_align_block_size(ti, 16, 16)]

    got = calls()
    assert not isinstance(pkg._lib.fast(), type(no_native_module))
    monkeypatch.setattr(pkg._lib, "_fast", no_native_module)
    calls()  # (the native path takes the second call of a shape)
    assert all(torch.equal(a, b) for a, b in zip(got, calls()))


def _table(pkg, folder, tuning):
    T = pkg.tuning
    (folder / T.config_name(16, 256, 512, 32, T.device_name() if torch.cuda.is_available()
                            else "dev")).write_text(T.dump_table({8: tuning}))


def test_reload_tables(pkg, tmp_path):
    T = pkg.tuning
    a, b = T.Tuning(T.ALWAYS, 4, 2, 0), T.Tuning(0, 0, 0, 0)
    for want in (a, b):
        _table(pkg, tmp_path, want)
        T.reload_tables()
        name = T.device_name() if torch.cuda.is_available() else "dev"
        assert T.load_table(16, 256, 512, 32, name, tmp_path) == {8: want}


@pytest.mark.gpu
def test_reload_tables_reaches_the_native_path(pkg, synth, dev, tmp_path, monkeypatch):
    """A rewritten table decides the next call's dispatch (tiles in header[2])."""
    T = pkg.tuning
    shape = synth.LayerShape(E=16, topk=4, K=512, N=256, group=32)
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, 40, dev, seed=5)
    args = (x, w13, w2, s13, s2, tw, ti, 32)
    monkeypatch.setattr(T, "CONFIG_DIR", tmp_path)
    tiles = []
    for tuning in (T.Tuning(0, 15, 0, 64), T.Tuning(0, 0, 0, 64)):
        _table(pkg, tmp_path, tuning)
        T.reload_tables()
        pkg.fused_experts_w4a16(*args)
        assert pkg._lib.fast().fused(*args) is not None
        ws, off = pkg.workspace_tensor(x, ti, w13, w2, 32)
        tiles.append(int(ws[off[2] + 8: off[2] + 12].view(torch.int32).item()))
    T.reload_tables()
    assert tiles[0] < tiles[1] == int(torch.unique(ti).numel())


class _Counting:
    """The native module, counting what is registered."""

    def __init__(self, native):
        self.native, self.seen = native, []

    def __getattr__(self, name):
        if name.startswith("set_"):
            self.seen.append(name)
        return getattr(self.native, name)


def test_each_eager_buffer_is_shown_once(pkg):
    """Threads on one stream whose calls grow its buffer: what the pool shows
    last is what it holds, and nothing is shown for a buffer that is reused
    or belongs to a capture."""
    shown = {}
    count = [0]

    def on_eager(device, stream, buf):
        shown[stream] = buf
        count[0] += 1

    pool = pkg.w4a16_moe.WorkspacePool(
        alloc=lambda n, d: torch.empty(n, dtype=torch.uint8), on_eager=on_eager,
        on_clear=shown.clear)
    sizes = [400 + 7 * i for i in range(200)]

    def worker(k):
        for n in sizes[k::4]:
            pool.get("cuda:0", 5, n)
            pool.get("cuda:0", 5, 300)
            pool.get("cuda:0", 5, n, capture_id=9)

    threads = [threading.Thread(target=worker, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert shown[5] is pool.get("cuda:0", 5, 1) and shown[5].numel() == max(sizes)
    assert count[0] <= len(sizes)
    pool.clear()
    assert not shown


@pytest.mark.gpu
def test_declined_calls_register_nothing_again(pkg, synth, dev, monkeypatch):
    shape = synth.LayerShape(E=16, topk=4, K=512, N=256, group=32)
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, 6, dev, seed=8)
    odd = torch.zeros(6, 516, dtype=torch.bfloat16, device=dev)[:, :512]
    odd.copy_(x)
    native = pkg._lib.load_fast()
    native.clear_plans()
    pkg.w4a16_moe._WS_POOL.clear()
    counting = _Counting(native)
    monkeypatch.setattr(pkg._lib, "_fast", counting)
    t = pkg.Tuning()
    for i in range(3):  # declined for its row stride, and for its tuning
        a = pkg.fused_experts_w4a16(odd, w13, w2, s13, s2, tw, ti, 32)
        b = pkg.fused_experts_w4a16(x, w13, w2, s13, s2, tw, ti, 32, tuning=t)
        assert sorted(counting.seen) == ["set_plan", "set_workspace"], i
    assert torch.equal(_bits(native.fused(x, w13, w2, s13, s2, tw, ti, 32)), _bits(a))
    assert torch.equal(_bits(a), _bits(b))


@pytest.mark.gpu
def test_streams_threads_and_growth(pkg, synth, dev):
    """A stream seen for the first time goes through the Python path, which
    gives it a workspace; threads on streams of their own then run at once;
    a larger call grows the buffer both paths use."""
    shape = synth.LayerShape(E=16, topk=4, K=512, N=256, group=32)
    w = synth.make_weights(shape, dev, seed=1)
    ins = []
    for M in (8, 40, 300):
        x = synth.make_hidden(M, shape.K, dev, seed=M)
        tw, ti = synth.make_routing(M, shape.E, shape.topk, dev, seed=M)
        ins.append((x, *w, tw, ti, 32))
    pkg.w4a16_moe._WS_POOL.clear()  # stream handles come round again
    want = [pkg.fused_experts_w4a16(*a) for a in ins]
    torch.cuda.synchronize()
    bad, done = [], []

    def worker():
        try:
            calls()
            done.append(True)
        except Exception as err:  # (a thread's own ends with it)
            bad.append(repr(err))

    def calls():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            if pkg._lib.fast().fused(*ins[0]) is not None:
                bad.append("a new stream has no workspace")
            for _ in range(20):
                for a, e in zip(ins, want):
                    if not torch.equal(_bits(pkg.fused_experts_w4a16(*a)), _bits(e)):
                        bad.append("bits")
            ws, _ = pkg.workspace_tensor(ins[2][0], ins[2][6], w[0], w[1])
            if pkg._lib.fast().fused(*ins[2]) is None:
                bad.append("not taken")
        s.synchronize()

    threads = [threading.Thread(target=worker) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
    assert len(done) == len(threads)


@pytest.mark.gpu
def test_capture_uses_the_captures_own_workspace(pkg, synth, dev):
    shape = synth.LayerShape(E=16, topk=4, K=512, N=256, group=32)
    w13, w2, s13, s2, x, tw, ti = _make(synth, shape, 40, dev, seed=3)
    args = (x, w13, w2, s13, s2, tw, ti, 32)
    want = pkg.fused_experts_w4a16(*args)
    torch.cuda.synchronize()
    taken = []
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        taken.append(pkg._lib.fast().fused(*args))
        out = pkg.fused_experts_w4a16(*args)
    assert taken == [None]
    for _ in range(3):
        out.zero_()
        pkg.fused_experts_w4a16(*args)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(_bits(out), _bits(want))
    del g
    pkg.release_graph_workspaces()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 7, 900])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_router_and_align(pkg, dev, M, dtype):
    g = torch.Generator(device=dev).manual_seed(M)
    logits = torch.randn((M, 64), generator=g, device=dev).to(dtype)
    f = pkg._lib.fast()
    w, ids = f.router(logits, 10, True)
    w2, ids2 = torch.empty_like(w), torch.empty_like(ids)
    pkg.router_topk_softmax(logits, 10, out=(w2, ids2))  # the Python path
    assert torch.equal(w, w2) and torch.equal(ids, ids2)
    assert f.router(logits.t().contiguous().t(), 10, True) is None or M == 1
    with pytest.raises(pkg._lib.W4A16Error):
        pkg.router_topk_softmax(logits, 65)
    got = f.align(ids, 16, 64)
    want = pkg.moe_align_block_size_full(ids, 16, 64)[:3]
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert all(torch.equal(a, b) for a, b in zip(f.align(ids.to(torch.int64), 16, 64), want))
    with pytest.raises(pkg._lib.W4A16Error):
        pkg.moe_align_block_size(ids, 0, 64)
