"""out and lse of the plane-split forward with two units per wavefront where its rounds and its stream of tiles can go wrong: rounds of one to
eight units (four and fewer have one per wavefront), sweeps shorter than the tiles that are requested ahead, windows that end in the
middle of a tile, a last tile that the sequence does not fill, shares, both plane counts, and logits that leave the reference point of the
first tile behind (a unit's sums are brought to another one).  (Up to 32 columns, few deltas and short sequences: the same cases on the kernel
with one unit per wavefront; tests/test_routes.py says which.)  Against the fp32 FMA kernels (accurate expf and logf), to the bars of the
other tests of these kernels; lse to 1e-5 of its largest value (16 bits: of exact products of 16-bit inputs, the same)."""
import pytest
import torch

from oracle import simplicial_oracle as orc
from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu
BF, FP, F32 = torch.bfloat16, torch.float16, torch.float32
BAR = {BF: 1e-2, FP: 2e-3, F32: 1e-5}
TYPES = [(F32, 16), (F32, 32), (F32, 64), (BF, 40), (BF, 56), (BF, 72), (BF, 96), (FP, 48), (FP, 80)]


def _inputs(dtype, B, N, H, D, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [(torch.randn(B, N, H, D, generator=g, device="cuda") * (std if t < 3 else 1.0)).to(dtype) for t in range(5)]


@pytest.mark.parametrize("dtype,D", TYPES)
@pytest.mark.parametrize("B,N,H,w1,w2,bias,scale", [
    (1, 1, 1, 0, 0, 0.0, None), (1, 33, 1, 0, 0, 0.0, None), (1, 300, 2, 40, 0, 0.1, None), (2, 129, 1, 128, 3, 0.0, 0.2), (1, 97, 3, 31, 4, 0.0, None),
    (1, 200, 1, 500, 8, 0.2, None), (1, 161, 1, 3, 12, 0.0, -0.1), (1, 700, 40, 129, 5, 0.0, None), (1, 520, 2, 95, 33, -0.1, None), (3, 40, 5, 40, 39, 0.0, 0.0),
    (1, 640, 30, 70, 40, 0.0, None)])
def test_forward_matches_the_fma_kernels(dtype, D, B, N, H, w1, w2, bias, scale):
    import simplical_attn_amd as sa
    x = _inputs(dtype, B, N, H, D, N + D)
    out, lse = sa.simplicial_forward(*x, w1, w2, scale, bias, -bias)
    want, want_lse = sa.simplicial_forward(*x, w1, w2, scale, bias, -bias, flags=1)
    assert_close_rel(out, want.cpu(), BAR[dtype], "out")
    assert_close_rel(lse, want_lse.cpu(), 1e-5, "lse")
    assert torch.equal(out, sa.simplicial_forward(*x, w1, w2, scale, bias, -bias)[0])


@pytest.mark.parametrize("dtype,D", TYPES[2:])
@pytest.mark.parametrize("B,N,H,w1,w2,bias", [(1, 33, 150, 20, 20, 0.1), (2, 40, 80, 40, 39, 0.0), (1, 65, 90, 64, 11, -0.2), (3, 96, 33, 5, 9, 0.0), (1, 130, 70, 200, 15, 0.0)])
def test_short_sequences_of_many_heads(dtype, D, B, N, H, w1, w2, bias):
    """Sequences of two to five tiles, too many for the kernel with one unit per wavefront."""
    test_forward_matches_the_fma_kernels(dtype, D, B, N, H, w1, w2, bias, None)


@pytest.mark.parametrize("dtype,D", TYPES)
@pytest.mark.parametrize("heads,w2,bias", [(2, 12, 0.0), (40, 3, 0.0), (40, 20, 0.3)])
def test_logits_that_leave_the_reference_point_behind(dtype, D, heads, w2, bias):
    """Keys away from the queries' own tile have logits more than 64 octaves above it.  A row's largest logits
    decide it; they are off by 2^-24 of the sum of the products' magnitudes (here up to 2^10) per rounding, which lse shows (absolute)."""
    import simplical_attn_amd as sa
    x = _inputs(dtype, 1, 470, heads, D, D)
    x[0] = x[0].abs() + 0.5
    x[2] = x[2].abs() + 0.5
    ramp = torch.where(torch.arange(470, device="cuda") % 170 < 60, 3.0, -3.0)[None, :, None, None]
    x[1] = (ramp + 0.1 * x[1].float()).to(dtype)
    out, lse = sa.simplicial_forward(*x, 300, w2, 90.0 / D, bias, bias)
    want, want_lse = sa.simplicial_forward(*x, 300, w2, 90.0 / D, bias, bias, flags=1)
    assert torch.isfinite(out).all() and (lse.abs().max() > 100)
    assert_close_rel(lse, want_lse.cpu(), 2e-5, "lse")
    assert_close_rel(out, want.cpu(), max(BAR[dtype], 2e-3), "out")


@pytest.mark.parametrize("dtype,D", TYPES)
@pytest.mark.parametrize("std", [3.0, 4.0])
def test_widely_spread_logits(dtype, D, std):
    """Logits of standard deviation 27 and 64 on single rows: the reference point moves in some rows and not in others, first rows whose units
    have no key among them.  They are off by 2^-24 of the sum of the products' magnitudes (some 2^9) per rounding, and so are lse and, near
    ties, out."""
    import simplical_attn_amd as sa
    x = _inputs(dtype, 1, 400, 6, D, D, std)
    for w2 in (3, 20):
        out, lse = sa.simplicial_forward(*x, 150, w2)
        want, want_lse = sa.simplicial_forward(*x, 150, w2, flags=1)
        assert torch.isfinite(out).all()
        assert_close_rel(lse, want_lse.cpu(), 1e-5, "lse")
        assert_close_rel(out, want.cpu(), max(BAR[dtype], 1e-3), "out")


@pytest.mark.parametrize("dtype,D", [(F32, 64), (BF, 40), (BF, 56), (BF, 72), (BF, 96), (FP, 48), (FP, 96)])
@pytest.mark.parametrize("bias", [0.0, 0.25])
def test_the_reference_point_comes_off_the_logits_last(dtype, D, bias):
    """The queries' own tile holds logits of -5, one key before it a small generic one, which decides the row (all K' rows are the same, so that the
    nine deltas agree in every rounding).  Less the reference point it is
    7.2 octaves, where a rounding has a root mean square of 2^-22 / sqrt(12) octaves (1e-7 in lse): one of the difference, one of the scale
    where that is multiplied on last, and half of one for the logit's chain at its own size and lse itself.  With the reference point at the start of the chain
    all 12 to 36 roundings had that size (2.8e-7 to 4.5e-7 in lse)."""
    import simplical_attn_amd as sa
    g = torch.Generator().manual_seed(D)
    x = [torch.randn(2, 64, 70, D, generator=g) for _ in range(5)]
    x[0], x[2] = 0.5 * x[0], (0.5 * x[2][:, :1]).expand_as(x[2]).contiguous()
    x[0][..., 0], x[2][..., 0] = 1.0, 1.0 - bias
    key = x[1][:, 31].clone()
    x[1][:] = 0.0
    x[1][..., 0] = -5.0 * D ** 0.5
    key[..., 0] = 0.0
    x[1][:, 31] = key
    x = [t.to(dtype) for t in x]
    lse = sa.simplicial_forward(*[t.cuda() for t in x], 63, 8, None, bias)[1][:, :, 32:]
    want = orc.forward_windowed(*[t.double() for t in x], 63, 8, None, bias)[1][:, :, 32:]
    error = (lse.double().cpu() - want).pow(2).mean().sqrt().item()
    assert error < 2.3e-7, error


@pytest.mark.parametrize("dtype,D", [(F32, 64), (BF, 40), (BF, 56), (BF, 72), (BF, 96), (FP, 48), (FP, 80)])
@pytest.mark.parametrize("gap", [12.0, 30.0, 60.0, 1e3, 7e3, 1e6, 1e9, None])
@pytest.mark.parametrize("w2,bias", [(9, 0.0), (2, 0.0), (40, 0.25)])
def test_an_own_tile_far_below_the_other_keys(dtype, D, gap, w2, bias):
    """Keys from 64 on are masked by a large finite K row (`gap` octaves; None: their logits overflow to -inf), so that every row from there on
    has an own tile far below the logits that decide it.  Those logits have a size of up to 8: roundings of 2^-22 / sqrt(12) octaves, some three of them
    in lse, and to the usual bars in out."""
    import simplical_attn_amd as sa
    if dtype == FP and (gap is None or gap > 1e4):
        pytest.skip("no such K row in fp16")
    g = torch.Generator().manual_seed(D + w2)
    x = [torch.randn(2, 150, 8, D, generator=g) for _ in range(5)]
    size = 1.0 if gap is not None else 8.0
    x[0][..., 0], x[2][..., 0] = size, size - bias
    x[1][..., 0] = 0.0
    x[1][:, 64:] *= 0.1
    x[1][:, 64:, :, 0] = -3e38 if gap is None else -gap * 0.6931 * D ** 0.5
    x = [t.to(dtype) for t in x]
    out, lse = sa.simplicial_forward(*[t.cuda() for t in x], 149, w2, None, bias, -bias)
    want, want_lse = orc.forward_windowed(*[t.double() for t in x], 149, w2, None, bias, -bias)
    assert (lse.double().cpu() - want_lse)[:, :, 64:].pow(2).mean().sqrt() < 4.5e-7
    assert_close_rel(out[:, 64:], want[:, 64:], {F32: 3e-6}.get(dtype, BAR[dtype]), "out")


def _far_tile(dtype, D, own, far, size, heads=8, N=150):
    """Rows from 64 on: keys of the own tile at `own` octaves, those before at `far`; values v1 and v2 of a size"""
    g = torch.Generator().manual_seed(D)
    x = [torch.randn(2, N, heads, D, generator=g) for _ in range(5)]
    x[0][..., 0], x[2][..., 0] = 4.0, 4.0
    x[1] *= 0.1
    x[1][..., 0] = far * 0.6931 * D ** 0.5 / 16
    x[1][:, 64:, :, 0] = own * 0.6931 * D ** 0.5 / 16
    x[3], x[4] = x[3] * size, x[4] * size
    return [t.to(dtype) for t in x]


@pytest.mark.parametrize("dtype,D", [(F32, 64), (BF, 40), (BF, 56), (BF, 72), (BF, 96)])
@pytest.mark.parametrize("own,far,size", [(10.0, 45.0, 2.0 ** 52), (4.0, 40.0, 2.0 ** 46), (20.0, 50.0, 2.0 ** 56)])
@pytest.mark.parametrize("w2,heads", [(9, 8), (30, 1)])
def test_values_that_large_weights_would_make_infinite(dtype, D, own, far, size, w2, heads):
    """Weights of 2^30 to 2^36, relative to the own tile's, times products v1*v2 of 2^92 to 2^112 are no floats; the outputs are, and so are the
    sums over shares (one head), with weights up to 1: at most 150 * 31 products of 2^112 * 2^4, 2^128.2 if all had one sign."""
    import simplical_attn_amd as sa
    x = _far_tile(dtype, D, own, far, size, heads)
    out, lse = sa.simplicial_forward(*[t.cuda() for t in x], 149, w2)
    want, want_lse = orc.forward_windowed(*[t.double() for t in x], 149, w2)
    assert torch.isfinite(out).all() and want.abs().max() > 2.0 ** 90
    assert_close_rel(out, want, {F32: 1e-5}.get(dtype, BAR[dtype]), "out")
    assert_close_rel(lse, want_lse, 1e-5, "lse")


@pytest.mark.parametrize("dtype,D", [(F32, 64), (BF, 40), (BF, 56), (BF, 72), (BF, 96)])
@pytest.mark.parametrize("w2,heads", [(9, 8), (30, 1)])
def test_weights_far_below_the_epsilon(dtype, D, w2, heads):
    """Rows whose largest logit is at -125 octaves, 35 above the own tile: out is 2^(26.6 - 125) times the values' sums, which are large.  An octave is
    rounded at the size of 125 (2^-18: 3e-6 of a weight)."""
    import simplical_attn_amd as sa
    x = _far_tile(dtype, D, -160.0, -125.0, 2.0 ** 20, heads)
    out, lse = sa.simplicial_forward(*[t.cuda() for t in x], 149, w2)
    want, want_lse = orc.forward_windowed(*[t.double() for t in x], 149, w2)
    assert_close_rel(out[:, 70:], want[:, 70:], max(BAR[dtype], 3e-5), "out", atol=0.0)
    assert_close_rel(lse, want_lse, 1e-6, "lse")
