"""Rows of no whole number of 16-byte vectors (pointwise and row kernels) and several short
rows per wave, at the sizes where they can go wrong."""
import pytest
import torch
import torch.nn.functional as F

import tensorjit as tj
from parity import close_f32, close_lowp
from tensorjit import compiler as C
from tensorjit.backends import hip_backend as hb
from tensorjit.ir import DType, TensorType

DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def _close(out, ref, n=1):
    if out.dtype == torch.float32:
        close_f32(out, ref, scale=1e-5 * max(1.0, (n / 4096) ** 0.5))
    else:
        close_lowp(out, ref)


def test_short_rows_share_a_wave_and_long_ragged_rows_compile():
    def launch(fn, shapes, dt):
        src, (l,) = hb.generate(C.lower(tj.trace(fn, [TensorType(s, dt) for s in shapes]), "hip"))
        hb.compile_source(src, "gfx950")
        return src, l

    for n, lanes in [(8, 2), (64, 8), (72, 16), (256, 32)]:
        src, l = launch(tj.softmax, [(100000, n)], DType.bf16)
        rows = 256 // lanes
        assert l.grid == (-(-100000 // rows), 1, 1) and l.block == (256, 1, 1) and f"tj_group_sum<{lanes}>" in src
    _, l = launch(tj.softmax, [(1024, 64)], DType.bf16)
    assert l.grid == (128, 1, 1) and l.block == (64, 1, 1)           # too few rows for 4 waves each
    _, l = launch(tj.softmax, [(1023, 64)], DType.bf16)
    assert l.grid == (1023, 1, 1) and l.block == (64, 1, 1)          # fewer still: a wave per row
    # three row arrays of 14 chunks: the gain and the bias are loaded in their stage
    src, l = launch(lambda x, g, b: tj.layer_norm(x, g, b), [(64, 27691), (27691,), (27691,)], DType.bf16)
    assert "in0_r[14][8]" in src and "in1_r[" not in src and "tj_stv_u" in src


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("rows,n", [(1, 9), (5, 17), (70, 1001), (3, 4097), (2, 12001), (2, 32767), (1, 300001), (33, 63),
                                    (511, 9), (512, 9), (513, 1001), (512, 4097), (64, 32767)])
def test_ragged_rows_match_float64(dt, rows, n):
    """One element past and short of a vector, of a wave's chunks, of the 256 / 1024-lane
    layouts, and a split reduction: sums count the last chunk's shared elements once."""
    gen = torch.Generator(device=DEV).manual_seed(n)
    x = (torch.randn(rows, n, device=DEV, generator=gen) + 0.5).to(dt)
    g = (1 + 0.1 * torch.randn(n, device=DEV, generator=gen)).to(dt)
    X, G = x.double(), g.double()
    _close(tj.jit(lambda a, b: tj.layer_norm(a, b, b))(x, g), F.layer_norm(X, (n,), G, G), n)
    _close(tj.jit(lambda a: tj.softmax(a))(x), torch.softmax(X, -1), n)
    _close(tj.jit(lambda a: tj.mean(a * a, axis=-1))(x), (X * X).mean(-1), n)
    assert torch.equal(tj.jit(lambda a: tj.max(a, axis=-1))(x), x.amax(-1))
    _close(tj.jit(lambda a, b: a * b + tj.sigmoid(b))(x, g), X * G + torch.sigmoid(G), 1)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
def test_long_odd_row_split_over_workgroups(dt):
    """One row past the size from which a few rows take unaligned vectors."""
    n = (16 << 20) // torch.empty((), dtype=dt).element_size() + 3
    gen = torch.Generator(device=DEV).manual_seed(n)
    x = (torch.randn(1, n, device=DEV, generator=gen) + 0.5).to(dt)
    _close(tj.jit(lambda a: tj.mean(a, axis=-1))(x), x.double().mean(-1), n)
    assert torch.equal(tj.jit(lambda a: tj.max(a, axis=-1))(x), x.amax(-1))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [*DTYPES, torch.int32])
@pytest.mark.parametrize("shape,other", [((4096, 33), (33,)), ((7, 9, 13), (9, 1)), ((5, 8, 9), (5, 1, 9)), ((1000, 1001), (1001,))])
def test_ragged_pointwise_rows_are_exact(dt, shape, other):
    """Row-broadcast, column-broadcast and middle-broadcast operands over odd rows: small
    integers, every value exact; the last vector of a row overlaps its neighbour."""
    gen = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randint(-8, 9, shape, device=DEV, generator=gen).to(dt)
    y = torch.randint(-8, 9, other, device=DEV, generator=gen).to(dt)
    assert torch.equal(tj.jit(lambda a, b: a * b + a)(x, y), x * y + x)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("rows,n", [(4097, 2), (1025, 8), (33000, 24), (2049, 33), (5000, 64), (70001, 72), (1030, 127), (9001, 256)])
def test_short_rows_match_float64(dt, rows, n):
    """2-32 lanes per row, rows that do not fill the last wave or workgroup, ragged ones."""
    gen = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(rows, n, device=DEV, generator=gen).to(dt)
    g = (1 + 0.1 * torch.randn(n, device=DEV, generator=gen)).to(dt)
    X, G = x.double(), g.double()
    _close(tj.jit(lambda a: tj.softmax(a))(x), torch.softmax(X, -1))
    _close(tj.jit(lambda a, b: tj.rms_norm(a, b))(x, g), X * torch.rsqrt((X * X).mean(-1, keepdim=True) + 1e-6) * G)
    assert torch.equal(tj.jit(lambda a: tj.max(a, axis=-1))(x), x.amax(-1))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4096, 4099])
def test_fp16_stores_round_to_nearest_even(n):
    """Products of fp16 values rounded back to fp16: ties, subnormals, overflows to infinity and
    NaN come out with torch's bits."""
    bits = torch.arange(-(1 << 15), 1 << 15, device="cuda", dtype=torch.int32).to(torch.int16).view(torch.float16)
    a = bits[torch.randperm(1 << 16, device="cuda")][:n * 15].reshape(15, n)
    b = bits[torch.randperm(1 << 16, device="cuda")][:n * 15].reshape(15, n)
    out, ref = tj.jit(lambda x, y: x * y)(a, b), (a.float() * b.float()).half()
    nan = ref.isnan()
    assert torch.equal(out.isnan(), nan)
    assert torch.equal(out.view(torch.int16)[~nan], ref.view(torch.int16)[~nan])
