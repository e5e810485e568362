"""Attention of few queries or few heads: edges of the key blocks, the waves and the key splits."""
from __future__ import annotations

import re

import pytest
import torch

import tensorjit as tj
from tensorjit.backends import hip_backend as hb
from tensorjit.backends.hip_attention import _split_tile_lines, few_query_splits, fuse_attention
from tensorjit.compiler import lower
from tensorjit.ir import DType, TensorType


def attention(scale):
    return lambda q, k, v: tj.matmul(tj.softmax(tj.matmul(q, tj.transpose(k, -1, -2)) * scale), v)


def launches_of(shapes, dt=DType.bf16):
    p = fuse_attention(lower(tj.trace(attention(0.1), [TensorType(s, dt) for s in shapes]), "hip"))
    return hb.generate(p)


@pytest.mark.parametrize("dt", [DType.bf16, DType.f16])
@pytest.mark.parametrize("Sq,Sk,D,Dv", [(1, 1, 32, 32), (16, 4096, 96, 128), (4, 130, 64, 32)])
def test_few_queries_compile_and_keep_in_their_buffers(Sq, Sk, D, Dv, dt):
    src, launches = launches_of([(3, Sq, D), (3, Sk, D), (3, Sk, Dv)], dt)
    m = launches[0].meta
    assert m["schedule"] == "few-queries" and launches[0].grid == (3 * m["splits"], 1, 1)
    assert len(launches) == (2 if m["splits"] > 1 else 1)
    if m["splits"] > 1:
        assert m["workspace"] == m["splits"] * 3 * Sq * (Dv + 2) * 4
    assert m["lds_bytes"] <= 80 * 1024          # two workgroups per CU
    assert len(hb.compile_source(src, "gfx950")) > 1000


def test_seventeen_queries_and_a_forced_schedule_keep_the_tiled_kernels(monkeypatch):
    shapes = lambda n: [(3, n, 64), (3, 200, 64), (3, 200, 64)]  # noqa: E731
    assert launches_of(shapes(17))[1][0].meta["schedule"] == "double-buffer"
    monkeypatch.setenv("TENSORJIT_HIP_ATTENTION_WAVES", "4")
    assert launches_of(shapes(1))[1][0].meta["schedule"] == "double-buffer"


def test_partials_lie_in_the_streams_workspace():
    """Both launches of a split call, few queries and tiled, get the same per-stream memory."""
    from tensorjit.runtime import hip as rt
    for shapes in ([(320, n, 64) for n in (1, 1500, 1500)], [(8, n, 128) for n in (500, 1450, 1450)]):
        _, launches = launches_of(shapes)
        for launch in launches:
            launch.meta["kernel"] = 0
        layout, arena = hb.workspace_layout(launches, 512)
        refs = hb.launch_args(launches, [[]], layout)
        assert arena == 512 and not layout
        assert refs[0] == refs[1] == [(rt.WORKSPACE, hb.WS_ALIGN, launches[0].meta["workspace"])]


def test_every_split_has_a_block():
    for batch in (1, 3, 8, 100, 320, 512, 5000):
        for Sk in (1, 31, 32, 33, 127, 1000, 1025, 4000, 8191):
            for d in (32, 64, 128):
                blocks = -(-Sk // 32)
                n = few_query_splits(batch, Sk, d, d)
                per = -(-blocks // n)
                assert 1 <= n <= 32 and (n == 1 or blocks >= 4 * n)
                used = -(-blocks // per)
                assert (used - 1) * per < blocks <= used * per


@pytest.mark.parametrize("heads,Sq,Sk,D", [(32, 1, 1500, 64), (16, 1, 1000, 128)])
def test_the_hosts_time_counts_only_for_a_program_of_one_kernel(heads, Sq, Sk, D):
    """8 us of kernel in one part hide behind the host's launch of a lone call, and not between
    the other kernels of a program (in a captured graph, us: 8.4 in one part, 5.3 in six)."""
    assert few_query_splits(heads, Sk, D, D) == 1 and few_query_splits(heads, Sk, D, D, alone=False) > 3
    shapes = [(heads, n, D) for n in (Sq, Sk, Sk)]
    assert launches_of(shapes)[1][0].meta["splits"] == 1
    fn = lambda q, k, v, w: tj.matmul(attention(0.1)(q, k, v), w)  # noqa: E731
    p = fuse_attention(lower(tj.trace(fn, [TensorType(s, DType.bf16) for s in (*shapes, (D, D))]), "hip"))
    assert [k.kind for k in p.kernels] == ["attention", "matmul"]
    assert hb.generate(p)[1][0].meta["splits"] > 3


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,splits,scale", [
    ((1, 2, 1, 1, 32, 32), None, 0.2), ((2, 3, 16, 31, 64, 128), None, 0.1), ((1, 5, 3, 32, 96, 32), None, 0.1),
    ((2, 2, 7, 129, 128, 96), None, -0.1), ((1, 4, 1, 2050, 128, 128), "5", 0.09), ((1, 1, 16, 4097, 64, 64), None, 0.125),
    ((3, 100, 2, 260, 64, 64), "2", 0.125)])
def test_few_queries_match_fp32_attention(shape, splits, scale, dt, monkeypatch):
    """The bound: P is rounded to 16 bits (2^-9 / 2^-11 of each weight), the output once more."""
    if splits:
        monkeypatch.setenv("TENSORJIT_HIP_ATTENTION_SPLITS", splits)
    B, H, Sq, Sk, D, Dv = shape
    gen = torch.Generator(device="cuda").manual_seed(Sk)
    q, k, v = [torch.randn(B, H, n, d, device="cuda", generator=gen).to(dt) for n, d in ((Sq, D), (Sk, D), (Sk, Dv))]
    print(f"few queries {shape} {splits} {dt}", flush=True)
    f = tj.jit(attention(scale))
    out = f(q, k, v)
    assert f.compiled(q, k, v).launches[0].meta["schedule"] == "few-queries"
    p = torch.softmax(torch.matmul(q.cpu().double(), k.cpu().double().transpose(-1, -2)) * scale, -1)
    ref = torch.matmul(p, v.cpu().double())
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    bound = eps * (torch.matmul(p, v.cpu().double().abs()) + ref.abs()) + 1e-6
    assert bool(((out.cpu().double() - ref).abs() <= bound).all())


def test_shares_of_the_key_blocks_cover_them():
    """Key splits of the tiled schedule that do not divide the blocks: the emitted first blocks
    and the guarded last one give every block to exactly one split."""
    for KB in range(2, 70):
        for n in (n for n in range(2, 33) if KB // n >= 2):
            KBL = -(-KB // n)
            lines = " ".join(_split_tile_lines(2, 3, n, KB, "unsigned int"))
            expr = re.search(r"kb0 = (.*?);", lines).group(1)
            m = re.fullmatch(r"sp \* (\d+)u(?: - \(sp > (\d+)u \? sp - \2u : 0u\))?", expr)
            assert int(m.group(1)) == KBL
            long = int(m.group(2)) if m.group(2) else n
            seen = [sp * KBL - max(0, sp - long) + j for sp in range(n) for j in range(KBL if sp < long else KBL - 1)]
            assert seen == list(range(KB)), (KB, n)


@pytest.mark.parametrize("shapes,splits", [
    ([(8, 1100, 128)] * 3, 3), ([(8, 1450, 128)] * 3, 2), ([(64, 330, 64)] * 3, 1), ([(32, 600, 128)] * 3, 1)])
def test_key_splits_reach_idle_compute_units_only(shapes, splits):
    assert launches_of(shapes)[1][0].meta["splits"] == splits


@pytest.mark.gpu
@pytest.mark.parametrize("shape,splits", [((2, 100, 300, 64, 64), "2"), ((3, 129, 448, 128, 128), "3"),
                                          ((2, 40, 833, 64, 128), "4"), ((1, 260, 1025, 96, 32), "5")])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_uneven_key_splits_match_fp32_attention(shape, splits, dt, monkeypatch):
    """5 blocks in 2 parts (ragged), 7 in 3, 14 in 4 (ragged), 17 in 5 (one key in the last block)."""
    monkeypatch.setenv("TENSORJIT_HIP_ATTENTION_SPLITS", splits)
    B, Sq, Sk, D, Dv = shape
    gen = torch.Generator(device="cuda").manual_seed(Sk)
    q, k, v = [torch.randn(B, n, d, device="cuda", generator=gen).to(dt) for n, d in ((Sq, D), (Sk, D), (Sk, Dv))]
    print(f"uneven splits {shape} {splits} {dt}", flush=True)
    f = tj.jit(attention(0.1))
    out = f(q, k, v)
    assert f.compiled(q, k, v).launches[0].meta["splits"] == int(splits)
    p = torch.softmax(torch.matmul(q.cpu().double(), k.cpu().double().transpose(-1, -2)) * 0.1, -1)
    ref = torch.matmul(p, v.cpu().double())
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    bound = eps * (torch.matmul(p, v.cpu().double().abs()) + ref.abs()) + 1e-6
    assert bool(((out.cpu().double() - ref).abs() <= bound).all())


@pytest.mark.gpu
def test_blocks_of_minus_infinity_scores_add_nothing():
    """Leading keys whose scores are -inf (a whole wave's blocks among them) weigh zero."""
    q = torch.ones(1, 1, 1, 32, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros(1, 1, 200, 32, device="cuda", dtype=torch.bfloat16)
    k[:, :, :150] = -torch.inf
    v = torch.randn(1, 1, 200, 32, device="cuda").bfloat16()
    out = tj.jit(attention(1.0))(q, k, v)
    torch.testing.assert_close(out[0, 0, 0].float(), v[0, 0, 150:].float().mean(0), atol=2e-3, rtol=8e-3)
