"""Column reductions over narrow rows (several rows per workgroup pass, the last workgroup
finishes) and over rows of no whole number of 16-byte vectors."""
import pytest
import torch

import tensorjit as tj
from parity import close_f32, close_lowp
from tensorjit import compiler as C
from tensorjit.backends import hip_backend as hb
from tensorjit.backends import hip_kernels as hk
from tensorjit.ir import DType, TensorType

DEV = "cuda:0"


def test_narrow_rows_fold_over_the_leading_axis_only():
    def kinds(shape, axis):
        p = C.lower(tj.trace(lambda x: tj.sum(x, axis=axis), [TensorType(shape)]), "hip")
        return [k.kind for k in hb.fold_transpose_into_reduce(p).kernels]

    assert kinds((1000, 16), 0) == ["colreduce"] and kinds((4, 300, 96), 1) == ["copy", "reduce"]
    assert kinds((1000, 127), 0) == kinds((1000, 129), 0) == ["colreduce"]


@pytest.mark.parametrize("Rd,L", [(1, 1), (5, 3), (96, 8), (4096, 31), (618418, 18), (1 << 20, 1), (257, 127)])
def test_narrow_layout_covers_every_row_once(Rd, L):
    S, RS = hk.col_narrow_layout(Rd, L, Rd * L * 16)
    assert S >= 1 and (S - 1) * RS < Rd <= S * RS and S <= hk.COL_MAX_SPLITS
    G = hk.COL_NARROW_LANES // L
    rows = sorted(j for s in range(min(S, 3)) for gi in range(G) for j in range(s * RS + gi, min((s + 1) * RS, Rd), G))
    assert rows == list(range(min(min(S, 3) * RS, Rd)))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16, torch.int32])
@pytest.mark.parametrize("shape,axis", [((1, 7), 0), ((5, 3), 0), ((1000, 1), 0), ((4097, 31), 0), ((70001, 72), 0),
                                        ((3000, 127), 0), ((64, 3, 8), 0), ((600, 1139), 0), ((3, 500, 333), 1),
                                        ((100, 17, 129), 0)])
def test_column_reductions_are_exact_on_integers(dt, shape, axis):
    """Narrow and ragged rows, one slice and many, twice each (the counter is back at zero):
    small integers, every partial exact; maxima of the same."""
    gen = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randint(-3, 4, shape, device=DEV, generator=gen).to(dt)
    f = tj.jit(lambda t: (tj.sum(t, axis=axis), tj.max(t * 2.0, axis=axis)))
    if len(shape) == 2:
        assert all(l.meta["family"].startswith("colreduce") for l in f.compiled(x).launches)
    for _ in range(2):
        s, m = f(x)
        assert torch.equal(s, x.double().sum(axis).to(dt)) and torch.equal(m, (x * 2).amax(axis))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(70001, 72), (5896, 1139), (300000, 5)])
def test_narrow_and_ragged_columns_match_float64(shape):
    """A folded prologue with a row-broadcast operand, a mean and an epilogue."""
    gen = torch.Generator(device=DEV).manual_seed(2)
    for dt in (torch.float32, torch.bfloat16):
        x = torch.randn(shape, device=DEV, generator=gen).to(dt)
        g = torch.randn(shape[1], device=DEV, generator=gen).to(dt)
        out = tj.jit(lambda t, w: tj.mean(tj.exp(t) * w, axis=0) + w)(x, g)
        # the plan computes the elementwise prologue in its own kernel when it is not folded:
        # either way one rounding of 16-bit intermediates per element, averaged over the rows
        ref = (x.double().exp() * g.double()).mean(0) + g.double()
        close_f32(out, ref, scale=1e-5 * (shape[0] / 64) ** 0.5) if dt == torch.float32 else close_lowp(out, ref)
