"""The workspace of products split over K: whose block a launch gets (a stream's, a captured
graph's, an exec's captured ahead), that blocks come back, and that calls do not wait."""
import ctypes
import gc

import pytest
import torch
from test_ring_gemm import DEV, _fn, _integers, _native, _ring

import tensorjit as tj
from tensorjit.ir import DType

pytestmark = pytest.mark.gpu

DT = DType.bf16


def _split_program(m=48, n=512, k=3072, split=4, seed=0, tile=(32, 64)):
    args, ref = _integers(m, n, k, True, DT, seed=seed)
    prog = _native(_fn(True), args, _ring(*tile, 4, 2, 2, 4, split, DT))
    assert prog is not None
    return prog, args, ref, torch.empty_like(ref)


def _ptrs(args, out):
    return [t.data_ptr() for t in args], [out.data_ptr()]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def test_recaptured_graphs_give_their_blocks_back():
    prog, args, ref, out = _split_program()
    prog.run(*_ptrs(args, out), _stream())
    for i in range(6):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            prog.run(*_ptrs(args, out), _stream())
        for _ in range(2):
            out.fill_(7)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref), i
        del graph
        gc.collect()
        torch.cuda.synchronize()
    assert prog.stats()["workspace_blocks"] <= 3         # the eager stream's, one graph's, one on its way back


def test_graphs_of_one_program_and_eager_calls_overlap():
    """Two live captured graphs and an eager stream, without any ordering between them."""
    prog, args, ref, out = _split_program()
    more = [_integers(48, 512, 3072, True, DT, seed=s) for s in (1, 2)]
    outs = [torch.empty_like(ref) for _ in more]
    graphs = []
    for (a, _), o in zip(more, outs):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            for _ in range(8):
                prog.run(*_ptrs(a, o), _stream())
    streams = [torch.cuda.Stream() for _ in range(3)]
    for _ in range(4):
        for t in (out, *outs):
            t.fill_(7)
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
        for _ in range(8):
            prog.run(*_ptrs(args, out), streams[2].cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and all(torch.equal(o, r) for o, (_, r) in zip(outs, more))
    assert prog.stats()["workspace_blocks"] == 3


@pytest.mark.parametrize("heads,Sq,Sk,D", [(320, 1, 1500, 64), (8, 500, 1450, 128)])
def test_key_split_attention_on_several_streams(heads, Sq, Sk, D):
    """A lone attention call, split over its keys by a rule on its sizes, on three streams
    without any ordering between them: bit-equal to calls one after the other."""
    fn = tj.jit(lambda q, k, v: tj.matmul(tj.softmax(tj.matmul(q, tj.transpose(k, -1, -2)) * D ** -0.5), v), tune=False)
    gen = torch.Generator(device=DEV).manual_seed(heads)
    cases = [[torch.randn(heads, n, D, device=DEV, generator=gen).half() for n in (Sq, Sk, Sk)] for _ in range(3)]
    cp = fn.compiled(*cases[0])
    assert cp.launches[0].meta["splits"] > 1 and cp.native.arena()[1] == 0
    refs = [fn(*c).clone() for c in cases]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in cases]
    got = [[] for _ in cases]
    for _ in range(10):
        for s, c, g in zip(streams, cases, got):
            with torch.cuda.stream(s):
                g.append(fn(*c))
    torch.cuda.synchronize()
    assert all(torch.equal(o, ref) for ref, g in zip(refs, got) for o in g)


def test_first_call_on_a_stream_returns_while_the_stream_is_busy():
    prog, args, ref, out = _split_program()
    prog.run(*_ptrs(args, out), _stream())               # the block allocated with the program is taken
    a = torch.randn(8192, 8192, device=DEV, dtype=torch.bfloat16)
    torch.mm(a, a)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    out.fill_(7)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(60):                              # some 50 ms
            torch.mm(a, a)
    prog.run(*_ptrs(args, out), side.cuda_stream)
    assert not side.query()
    side.synchronize()
    assert torch.equal(out, ref) and prog.stats()["workspace_blocks"] == 2


def test_exec_captured_ahead_serves_the_stream_that_replays_it():
    prog, args, ref, out = _split_program()
    prog.capture(*_ptrs(args, out))
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    for s, captures in ((a, 1), (a, 1), (b, 2), (a, 2), (b, 2)):
        out.fill_(7)
        torch.cuda.synchronize()
        prog.replay(*_ptrs(args, out), s.cuda_stream)
        s.synchronize()
        assert torch.equal(out, ref) and prog.stats()["graph_captures"] == captures


def test_replayed_program_of_many_split_launches_on_several_streams():
    """Twelve split products replay as a graph by default; the streams' execs do not share
    partials or counters."""
    fn = tj.jit(lambda w, *xs: tuple(tj.linear(x, w) for x in xs), tune=False)
    sets = []
    for seed in range(3):
        gen = torch.Generator(device=DEV).manual_seed(seed)
        r = lambda *s: torch.randint(-2, 3, s, device=DEV, generator=gen).to(torch.bfloat16)  # noqa: E731
        w, xs = r(256, 6144), [r(32, 6144) for _ in range(12)]
        sets.append((w, xs, [(x.double() @ w.double().t().contiguous()).to(torch.bfloat16) for x in xs]))
    cp = fn.compiled(sets[0][0], *sets[0][1])
    assert cp.use_graph and len(cp.launches) >= 12 and all(c.KSPLIT > 1 for c in cp.matmul_configs.values())
    streams = [torch.cuda.Stream() for _ in sets]
    torch.cuda.synchronize()
    for _ in range(6):
        got = []
        for s, (w, xs, _) in zip(streams, sets):
            with torch.cuda.stream(s):
                got.append(fn(w, *xs))
        torch.cuda.synchronize()
        for outs, (_, _, refs) in zip(got, sets):
            assert all(torch.equal(o, r) for o, r in zip(outs, refs))
        del got, outs
    assert cp.stats["graph_replays"] >= 9 and cp.native_stats()["workspace_blocks"] <= 3


@pytest.mark.parametrize("k", [192, 6144])               # without and with K splits
def test_replayed_program_is_recorded_in_the_callers_capture(k):
    """A program that replays graphs of its own, called under stream capture: its launches are
    part of the captured graph, and eager calls on that stream stay right afterwards."""
    fn = tj.jit(lambda w, *xs: tuple(tj.linear(x, w) for x in xs), tune=False)
    gen = torch.Generator(device=DEV).manual_seed(0)
    r = lambda *s: torch.randint(-2, 3, s, device=DEV, generator=gen).to(torch.bfloat16)  # noqa: E731
    w, xs = r(256, k), [r(32, k) for _ in range(12)]
    refs = [(x.double() @ w.double().t().contiguous()).to(torch.bfloat16) for x in xs]
    assert fn.compiled(w, *xs).use_graph
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        outs = fn(w, *xs)
    for _ in range(3):
        for o in outs:
            o.fill_(7)
        graph.replay()
        with torch.cuda.stream(side):
            eager = fn(w, *xs)
        torch.cuda.synchronize()
        assert all(torch.equal(o, t) and torch.equal(e, t) for o, e, t in zip(outs, eager, refs))


def test_values_dropped_inside_a_capture_stay_the_graphs():
    """An intermediate dropped while capturing is written again by every replay: later calls on
    that stream, and on others, must not be given its memory."""
    f, g = tj.jit(lambda x: x * 2.0 + 1.0, tune=False), tj.jit(lambda x: tj.sigmoid(x), tune=False)
    x, other = torch.randn(257, 96, device=DEV), torch.randn(257, 96, device=DEV)
    want_f, want_g = f(other).clone(), g(f(x)).clone()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        y = f(x)
        z = g(y)
        del y
    for _ in range(3):
        with torch.cuda.stream(side):
            kept = [f(other) for _ in range(3)]
        kept += [f(other) for _ in range(3)]
        torch.cuda.synchronize()
        z.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, want_g) and all(torch.equal(k, want_f) for k in kept)


def test_more_streams_than_blocks():
    prog, args, ref, _ = _split_program()
    outs = [torch.empty_like(ref) for _ in range(45)]
    hip = ctypes.CDLL("libamdhip64.so.7")
    streams = []
    for _ in outs:
        s = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
        streams.append(s)
    torch.cuda.synchronize()
    for o, s in zip(outs, streams):
        prog.run(*_ptrs(args, o), s.value)
    torch.cuda.synchronize()
    assert all(torch.equal(o, ref) for o in outs)
    assert prog.stats()["workspace_blocks"] <= 40
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0


def test_a_program_holds_one_block_until_a_second_stream_needs_one():
    """And run_static works from the static array and counters of its own, also as the program's
    first call and under capture."""
    m, n, split = 256, 4096, 4
    _split_program()                                     # the library's static array is in place
    args, ref = _integers(m, n, 4096, True, DT)
    out = torch.empty_like(ref)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    prog = _native(_fn(True), args, _ring(64, 64, 4, 2, 2, 4, split, DT))
    used = before - torch.cuda.mem_get_info()[0]
    ws = split * m * n * 4
    assert prog.stats()["workspace_blocks"] == 1 and used < 2 * ws, (used, ws)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        prog.run_static(*_ptrs(args, out), _stream())
    for _ in range(3):
        out.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
        out.fill_(7)
        prog.run_static(*_ptrs(args, out), _stream())
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
    assert prog.stats()["workspace_blocks"] == 1
