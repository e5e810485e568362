"""Where the rules for rows of no whole number of vectors draw their lines: pointwise kernels from
a MB, column splits of 16-bit and fp32 rows; results on both sides."""
import pytest
import torch

import tensorjit as tj
from parity import close_f32, close_lowp
from tensorjit import compiler as C
from tensorjit.backends import hip_backend as hb
from tensorjit.backends import hip_kernels as hk
from tensorjit.ir import DType, TensorType

DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


@pytest.mark.parametrize("dt", [DType.f32, DType.bf16])
def test_pointwise_rows_take_unaligned_vectors_from_a_megabyte(dt):
    n = 33
    last = (1 << 20) // (n * dt.itemsize)                      # rows below a MB
    for rows, unaligned in ((last, 0), (last + 1, 16 // dt.itemsize)):
        p = C.lower(tj.trace(lambda x, b: x + b, [TensorType((rows, n), dt), TensorType((n,), dt)]), "hip")
        _, (launch,) = hb.generate(p)
        assert launch.meta["family"] == "pointwise" and launch.meta["unaligned"] == unaligned


@pytest.mark.parametrize("itemsize", [2, 4])
@pytest.mark.parametrize("Rd,B", [(1, 9), (1141, 9), (4096, 9), (4097, 9), (6109, 172), (25133, 58), (395258, 10), (1 << 20, 4)])
def test_narrow_columns_split_few_times_and_cover_every_row(Rd, B, itemsize):
    L = -(-B // (16 // itemsize))
    S, RS = hk.col_narrow_layout(Rd, L, Rd * B * itemsize, itemsize)
    assert (S - 1) * RS < Rd <= S * RS
    if itemsize == 2:
        assert S <= 128 and (S == 1) == (Rd <= 32 * (256 // L))


def test_unaligned_wide_columns_split_fewer_times():
    for A, Rd, B, most in [(1, 12769, 498, 256), (3, 4286, 445, 128), (1, 9692, 316, 256)]:
        nb, RS, S = hk.col_layout(A, Rd, B, 8, 0, few=True, itemsize=2)
        assert S <= most < hk.col_layout(A, Rd, B, 8)[2] and (S - 1) * RS < Rd <= S * RS
    assert hk.col_layout(29, 43, 2893, 4, 0, few=True)[2] == 1 < hk.col_layout(29, 43, 2893, 4)[2]


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("rows,n", [(70001, 9), (20003, 33), (1100, 1001), (3, 200001), (5000, 14)])
def test_unaligned_pointwise_matches_float64(dt, rows, n):
    """Row and column broadcasts beside whole operands; the last vector of a row moved back."""
    gen = torch.Generator(device=DEV).manual_seed(n)
    x, y = [torch.randn(rows, n, device=DEV, generator=gen).to(dt) for _ in range(2)]
    g, c = torch.randn(n, device=DEV, generator=gen).to(dt), torch.randn(rows, 1, device=DEV, generator=gen).to(dt)
    f = tj.jit(lambda x, y, g, c: (x * g + y * c, tj.sigmoid(x)))
    out, s = f(x, y, g, c)
    assert f.compiled(x, y, g, c).launches[0].meta["unaligned"] == (16 // x.element_size() if rows * n * x.element_size() >= 1 << 20 else 0)
    X, Y, G, Cc = (t.double() for t in (x, y, g, c))
    close = close_f32 if dt == torch.float32 else close_lowp
    close(out, X * G + Y * Cc)
    close(s, torch.sigmoid(X))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("shape,axis", [((1141, 9), 0), ((4096, 9), 0), ((4097, 9), 0), ((6109, 172), 0), ((25133, 58), 0),
                                        ((12769, 498), 0), ((3, 4286, 445), 1), ((29, 43, 2893), 1)])
def test_columns_are_exact_on_integers(dt, shape, axis):
    gen = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randint(-1, 2, shape, device=DEV, generator=gen).to(dt)
    f = tj.jit(lambda t: tj.sum(t, axis=axis))
    for _ in range(2):
        assert torch.equal(f(x), x.double().sum(axis).to(dt))
