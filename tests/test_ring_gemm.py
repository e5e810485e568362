"""The ring-schedule GEMM: which products it takes, and its results at the edges of tiles, of
K tiles and of K splits, on one stream and on several."""
import re

import pytest
import torch

import tensorjit as tj
from tensorjit import compiler as C
from tensorjit.backends import hip_backend as hb
from tensorjit.ir import DType, TensorType
from tensorjit.runtime.autotune import RING_TILES, MatmulConfig, ring_candidates

TORCH = {DType.bf16: torch.bfloat16, DType.f16: torch.float16, DType.f32: torch.float32}


def _ring(tm, tn, waves, wm, wn, stages, split, dt):
    return MatmulConfig(tm, tn, 128 // dt.itemsize, waves, wm, wn, 16, 1, 8, 0, 0, 0, split, 0, stages)


def _fn(tb):
    return (lambda x, w, b: tj.linear(x, w, b)) if tb else (lambda x, w, b: tj.matmul(x, w) + b)


def _program(m, n, k, tb, dt, lead=()):
    types = [TensorType((*lead, m, k), dt), TensorType((n, k) if tb else (k, n), dt), TensorType((n,), dt)]
    return C.lower(tj.trace(_fn(tb), types), "hip")


@pytest.mark.parametrize("dt", [DType.bf16, DType.f16, DType.f32])
@pytest.mark.parametrize("tb", [True, False])
def test_ring_takes_whole_chunks_and_compiles(dt, tb):
    vk = 16 // dt.itemsize
    cfg = _ring(32, 64, 4, 2, 2, 4, 1, dt)
    ok = lambda c, m, n, k: hb.config_ok(c, dt, _program(m, n, k, tb, dt).kernels[0].anchor)  # noqa: E731
    assert ok(cfg, 33, 5 * vk, 3 * vk) and ok(cfg, 1, vk, vk)
    assert not ok(cfg, 33, 40, 3 * vk + 1)                       # rows of K that start inside a chunk
    assert ok(cfg, 33, 5 * vk + 1, 64) == tb                     # NN: rows of N too
    split = _ring(32, 64, 4, 2, 2, 4, 3, dt)
    tk = cfg.TK
    assert ok(split, 33, 40, 3 * tk) and ok(split, 33, 40, 4 * tk + vk)     # parts of 2, 2 and 1 K tiles
    assert not ok(split, 33, 40, 2 * tk)                         # a part without a K tile
    assert not ok(split, 33, 40, 4 * tk)                         # 2, 2, 0
    p = _program(100, 520, 1032, tb, dt)
    for c in (cfg, split):
        src, launches = hb.generate(p, {0: c})
        assert ("split_ws" in launches[0].meta) == (c.KSPLIT > 1)
        hb.compile_source(src, "gfx950")


@pytest.mark.parametrize("tb", [True, False])
@pytest.mark.parametrize("m,n,k,split", [(1, 64, 5 * 64, 3), (1, 64, 4 * 64 + 8, 3), (40, 72, 7 * 64, 4), (40, 72, 200, 1)])
def test_k_tiles_past_the_end_keep_the_scalar_offset_in_range(m, n, k, tb, split):
    """Parts with fewer K tiles load tiles past K: all lanes out of range (zeros), and the
    scalar offset still below the operand's size, from which the range check may subtract it."""
    src, _ = hb.generate(_program(m, n, k, tb, DType.bf16), {0: _ring(32, 64, 4, 2, 2, 4, split, DType.bf16)})
    size = {op: int(r) for op, r in re.findall(r"rs([AB]) = __builtin_amdgcn_make_buffer_rsrc\(\(void\*\)[AB]b, \(short\)0, (\d+),", src)}
    per = -(-(-(-k // 64)) // split)
    blocks = re.findall(r"  \{\n((?:    const unsigned int k\w+ = [^\n]*\n)+)((?:    __builtin_amdgcn_raw_ptr_buffer_load_lds[^\n]*\n)+)", src)
    assert len(blocks) >= per                                    # every tile of a part (none is in a loop here)
    for head, loads in blocks:
        for ksp in range(split):
            env = {"kt0": ksp * per, "min": min}
            for name, expr in re.findall(r"const unsigned int (\w+) = ([^\n]*);", head):
                expr = re.sub(r"(\d+)u\b", r"\1", expr)
                expr = re.sub(r"(.*?) < (.*?) \? (.*) : (.*)", r"(\3) if (\1) < (\2) else (\4)", expr)
                env[name] = eval(expr, {}, env)
            kf = env.get("kf", env["kt"])
            assert env["kleft"] == max(0, k - kf * 64) if "kleft" in env else (kf + 1) * 64 <= k
            for op, soff in re.findall(r"\(rs([AB]),.*, \(int\)\((.*?)\), 0, 0\);", loads):
                assert eval(re.sub(r"(\d+)u\b", r"\1", soff), {}, env) < size[op], (op, ksp, kf)


def test_ring_candidates_are_valid_and_bounded():
    for m, n, k in [(1, 768, 768), (64, 4096, 4096), (257, 1000, 8192), (8192, 8192, 8192), (3, 16, 16)]:
        mm = _program(m, n, k, True, DType.bf16).kernels[0].anchor
        for c in ring_candidates(m, n, k, 1, 2):
            assert c.KSPLIT == 1 or -(-m // c.TM) * -(-n // c.TN) * c.KSPLIT <= 1024
            if hb.config_ok(c, DType.bf16, mm):
                src, (launch,) = hb.generate(_program(m, n, k, True, DType.bf16), {0: c})
                assert launch.meta["lds_bytes"] <= 160 * 1024 and launch.grid[2] == c.KSPLIT


@pytest.mark.parametrize("m,n,k,tb,lead,staged", [
    (8192, 8192, 8192, False, (), True), (4096, 4096, 16384, False, (), True), (16384, 4096, 4096, False, (), True),
    (512, 512, 512, False, (64,), True), (8192, 8192, 8200, True, (), True), (2048, 11008, 4104, True, (), True),
    (4096, 4095, 4104, True, (), True),
    (2048, 4096, 4096, False, (), False), (2048, 11008, 4096, False, (), False), (1000, 4096, 4104, True, (), False)])
def test_products_without_a_direct_tile_keep_the_256_wide_staged_ones(m, n, k, tb, lead, staged):
    """The choice without tuning, and what tuning may time: products of whole rounds of 256x256
    tiles, where the ring's 128x128 measured 4-30% slower, and ones where it is the faster."""
    dt = DType.bf16
    b = TensorType((*lead, k, n) if not tb else (n, k), dt)
    types = [TensorType((*lead, m, k), dt), b, TensorType((n,), dt)]
    (kernel,) = C.lower(tj.trace(_fn(tb), types), "hip").kernels
    cands = hb._candidates(kernel)
    assert any(c.PINGPONG and (c.TM, c.TN) == (256, 256) for c in cands) and any(c.STAGES for c in cands)
    cfg = hb.analytic_config(kernel)
    assert (cfg.PINGPONG > 0) == staged and (cfg.STAGES > 0) == (not staged), cfg
    top = sorted(cands, key=hb._rank(kernel, cands))[:6]
    assert any(c.STAGES for c in top) and (not staged or sum(c.PINGPONG > 0 for c in top) >= 2)


SHARED = [((64, 1), 4096, 4096), ((16, 4), 4096, 4096), ((32, 1), 11008, 4096), ((8, 16), 4096, 4096),
          ((128, 1), 1024, 1024), ((2, 1), 4096, 4096), ((32, 17), 1024, 4096)]


@pytest.mark.parametrize("lead,n,k", SHARED)
@pytest.mark.parametrize("dt", [DType.bf16, DType.f16])
def test_batches_with_a_shared_weight_take_tiles_of_their_few_rows(lead, n, k, dt):
    """A batch of a few rows each with one weight: the weight counts once, so that the tile
    decides and not a floor that every tiling shares (which chose 192x256 for one row)."""
    (kernel,) = _program(lead[-1], n, k, True, dt, lead[:-1]).kernels
    cfg = hb.analytic_config(kernel)
    assert cfg.STAGES and cfg.TM == 32, cfg
    costs = sorted(hb._rank(kernel, hb._candidates(kernel))(c) for c in hb._candidates(kernel))
    assert costs[0] < costs[1] or costs[1] < costs[-1] / 2       # the estimates differ


def test_products_with_a_direct_tile_time_no_staged_ones():
    (kernel,) = _program(2048, 4096, 4096, True, DType.bf16).kernels
    assert all(c.STAGES or c.DIRECT or c.SPLIT_K > 1 for c in hb._candidates(kernel))
    (kernel,) = _program(4096, 4096, 4096, False, DType.f32).kernels
    assert all(c.STAGES for c in hb._candidates(kernel))
    (kernel,) = _program(700, 1501, 520, True, DType.bf16).kernels      # odd N: stores one by one
    assert all(c.STAGES for c in hb._candidates(kernel))


@pytest.mark.parametrize("m,n,k,direct", [(4096, 4096, 4096, True), (4096, 4096, 512, True), (2048, 4096, 1024, True),
                                          (512, 3072, 768, False), (512, 768, 3072, False)])
def test_fp32_products_of_a_full_grid_take_direct_tiles(m, n, k, direct):
    """Direct-to-LDS tiles measured 3-9% ahead of the ring there, and far behind it short of tiles."""
    (kernel,) = _program(m, n, k, True, DType.f32).kernels
    cfg = hb.analytic_config(kernel)
    assert bool(cfg.DIRECT) == direct and bool(cfg.STAGES) == (not direct), cfg


@pytest.mark.parametrize("m,n,k", [(1004, 1728, 6912), (1831, 1280, 5120), (307, 1792, 7168)])
def test_fp32_products_keep_the_split_of_their_long_sums(m, n, k):
    """A split's sums are shorter: 7.4e-7 from 64 bits in one part at K 1728, 5.3e-7 in two.  All
    unsplit tilings add in one order (the same bits), so speed alone chooses among them."""
    (kernel,) = _program(m, n, k, True, DType.f32).kernels
    cands = hb._candidates(kernel)
    first = min(cands, key=hb._rank(kernel, cands, fitted=False))
    assert first.KSPLIT > 1 and hb.analytic_config(kernel) == first


def test_split_launches_share_the_workspace():
    """Counters at the head of the block, as many as any launch has; partials behind them."""
    dt = DType.bf16
    g = tj.trace(lambda x, w, v: tj.linear(tj.linear(x, w), v),
                 [TensorType((64, 1024), dt), TensorType((2048, 1024), dt), TensorType((512, 2048), dt)])
    p = C.lower(g, "hip")
    _, launches = hb.generate(p, {0: _ring(64, 64, 4, 2, 2, 4, 2, dt), 1: _ring(32, 32, 4, 2, 2, 4, 4, dt)})
    args = hb.launch_args(launches, [[], []], {})
    from tensorjit.runtime import hip as rt
    assert args[0] == [(rt.WORKSPACE, 0, 32 * 4), (rt.WORKSPACE, 256, 2 * 32 * 64 * 64 * 4)]
    assert args[1] == [(rt.WORKSPACE, 0, 32 * 4), (rt.WORKSPACE, 256, 4 * 32 * 32 * 32 * 4)]


def _counter(src):
    """(operation, limit, count of the last workgroup, whether the kernel stores to the counter)."""
    (op, limit, last), = re.findall(r"tj_last_ = (atomic\w+)\(&?cnt_p(?:\[ct_\])?, (\d+)u\) == (\d+)u", src)
    return op, int(limit), int(last), re.search(r"(\*cnt_p|cnt_p\[ct_\]) = ", src) is not None


@pytest.mark.parametrize("kernel", ["ring", "columns"])
def test_counters_return_to_zero_after_launches_that_overlap(kernel):
    """Two launches on one counter, their workgroups' arrivals and (if the kernel has one) the
    last one's later reset in every order: the counter ends at zero, so the next launch is right."""
    if kernel == "ring":
        src, _ = hb.generate(_program(64, 512, 1024, True, DType.bf16), {0: _ring(64, 64, 4, 2, 2, 4, 3, DType.bf16)})
    else:
        p = hb.fold_transpose_into_reduce(C.lower(tj.trace(lambda x: tj.sum(x, axis=0), [TensorType((700, 24), DType.f32)]), "hip"))
        src, (launch,) = hb.generate(p)
        assert launch.meta["splits"] > 1
    op, limit, last, stores = _counter(src)
    S = last + 1

    def orders(value, left, resets):
        if not any(left) and not resets:
            yield value
        for i in range(2):
            if left[i]:
                rest = [n - (j == i) for j, n in enumerate(left)]
                after = value + 1 if op == "atomicAdd" else 0 if value >= limit else value + 1
                yield from orders(after, rest, resets + (stores and value == last))
        if resets:
            yield from orders(0, left, resets - 1)

    if S > 3:                                     # every order of two launches of three: the rule does not depend on S
        limit, last, S = limit - S + 3, 2, 3
    assert set(orders(0, [S, S], 0)) == {0}


DEV = "cuda:0"


def _native(fn, args, cfg):
    p = C.lower(tj.trace(fn, [C.tensor_type_of(a) for a in args]), "hip")
    (k,) = p.kernels
    if not hb.config_ok(cfg, hb.compute_dtype(k.anchor), k.anchor):
        return None
    from tensorjit.runtime import hip as rt
    src, ls = hb.generate(p, {0: cfg})
    refs = [[(rt.INPUT, j) for j in range(len(k.inputs))] + [(rt.OUTPUT, 0)]]
    return rt.NativeHipProgram(0, hb.compile_source(src, hb.arch_of(0), target=hb.target_of(0)), [l.name for l in ls],
                               [(l.grid, l.block, 0) for l in ls], hb.launch_args(ls, refs, {}), 0, len(args), 1)


def _integers(m, n, k, tb, dt, lead=(), seed=0):
    """Operands in {-2..2}: every product and sum is exact in any order (bf16 outputs round
    the same exact value)."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s: torch.randint(-2, 3, s, device=DEV, generator=gen).to(TORCH[dt])  # noqa: E731
    a, b, bias = r(*lead, m, k), r(n, k) if tb else r(k, n), r(n)
    ref = (torch.matmul(a.double(), b.double().t().contiguous() if tb else b.double()) + bias.double()).to(TORCH[dt])
    return [a, b, bias], ref


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [DType.bf16, DType.f16, DType.f32])
@pytest.mark.parametrize("tb", [True, False])
def test_ring_gemm_is_exact_at_the_edges(dt, tb):
    """M one past and one short of tiles, N of one and several chunks, K short of a K tile,
    of the ring, and ragged; K splits with unequal parts.  Twice each: the split's counters
    are back at zero."""
    tiles = [(32, 32, 4, 2, 2, 4), *RING_TILES, (64, 64, 8, 2, 4, 4)]
    for i, (m, n, k) in enumerate([(1, 16, 16), (33, 136, 72), (63, 64, 1032), (129, 520, 264)]):
        args, ref = _integers(m, n, k, tb, dt, seed=i)
        out = torch.empty_like(ref)
        ran = 0
        for tm, tn, waves, wm, wn, stages in tiles:
            for split in (1, 3):
                prog = _native(_fn(tb), args, _ring(tm, tn, waves, wm, wn, stages, split, dt))
                for _ in range(2 if prog else 0):
                    out.fill_(77)
                    prog.run([t.data_ptr() for t in args], [out.data_ptr()], torch.cuda.current_stream().cuda_stream)
                    assert torch.equal(out, ref), (m, n, k, tm, tn, waves, split)
                    ran += 1
        assert ran >= 2 * len(tiles)


@pytest.mark.gpu
def test_ring_gemm_batched_and_epilogue_operand():
    """A batch of products with a shared weight, and the residual ``x + linear(x, w)``."""
    dt = DType.bf16
    args, ref = _integers(40, 72, 200, True, dt, lead=(3,))
    out = torch.empty_like(ref)
    for split in (1, 2):
        prog = _native(_fn(True), args, _ring(32, 64, 4, 2, 2, 4, split, dt))
        prog.run([t.data_ptr() for t in args], [out.data_ptr()], torch.cuda.current_stream().cuda_stream)
        assert torch.equal(out, ref)
    (x, w, _), _ = _integers(50, 96, 96, True, dt)
    want = (x.double() + x.double() @ w.double().t().contiguous()).to(torch.bfloat16)
    out = torch.empty_like(want)
    prog = _native(lambda x, w: x + tj.linear(x, w), [x, w], _ring(32, 32, 4, 2, 2, 4, 1, dt))
    prog.run([x.data_ptr(), w.data_ptr()], [out.data_ptr()], torch.cuda.current_stream().cuda_stream)
    assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("lead,n,k", [((64, 1), 512, 1024), ((16, 4), 264, 1000), ((8, 16), 512, 768), ((3, 300), 392, 192),
                                      ((2, 3, 1), 768, 768)])
@pytest.mark.parametrize("dt", [DType.bf16, DType.f16, DType.f32])
def test_batches_with_a_shared_weight_through_the_chosen_tile(lead, n, k, dt):
    args, ref = _integers(lead[-1], n, k, True, dt, lead=lead[:-1])
    fn = tj.jit(_fn(True), tune=False)
    assert torch.equal(fn(*args), ref) and torch.equal(fn(*args), ref), fn.compiled(*args).matmul_configs


@pytest.mark.gpu
def test_split_products_on_several_streams_and_in_captured_graphs():
    """One split program on three streams without any ordering between them, then captured on
    a side stream and replayed with eager calls and synchronisation in between: the streams'
    partials and counters are their own."""
    dt = DType.bf16
    fn = tj.jit(lambda x, w, b: tj.linear(x, w, b), tune=False)
    cases = [_integers(48, 512, 6144, True, dt, seed=s) for s in range(3)]
    cp = fn.compiled(*cases[0][0])
    assert cp.matmul_configs[0].STAGES and cp.matmul_configs[0].KSPLIT > 1
    streams = [torch.cuda.Stream() for _ in cases]
    torch.cuda.synchronize()
    got = [[] for _ in cases]
    for _ in range(20):
        for s, (args, _), g in zip(streams, cases, got):
            with torch.cuda.stream(s):
                g.append(fn(*args))
    torch.cuda.synchronize()
    for (_, ref), outs in zip(cases, got):
        assert all(torch.equal(o, ref) for o in outs)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        a, b = fn(*cases[0][0]), fn(*cases[1][0])
    for _ in range(3):
        a.zero_(), b.zero_()
        graph.replay()
        eager = fn(*cases[2][0])
        torch.cuda.synchronize()
        assert torch.equal(a, cases[0][1]) and torch.equal(b, cases[1][1]) and torch.equal(eager, cases[2][1])
