"""dQ, dK' and dV' of the K'-side kernel for wide K windows where its rounds and its stream of tiles can go wrong: wavefronts with
one unit or none in the last round, sweeps that begin or end in the middle of a tile and at a sequence that does not fill its last
one, K windows wider than the sequence, segments of deltas, the pre-pass's unit, q and dO rows that do not fit LDS.  Against the
fp32 FMA kernels on the same inputs; the products, weights and dS are rounded to 16 bits in between, which the bar of the other
16-bit tests (2e-2 of the largest element, fp16 1.5e-2) covers."""
import pytest
import torch

from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu
BF, FP = torch.bfloat16, torch.float16


@pytest.mark.parametrize("dtype,B,N,H,D,w1,w2,bias", [
    (BF, 1, 2048, 1, 64, 330, 9, 0.0),      # the narrowest windows that are taken ...
    (BF, 1, 1100, 1, 128, 600, 9, 0.1),     # ... at both head_dims
    (FP, 2, 611, 2, 64, 2000, 7, 0.3),
    (BF, 1, 640, 40, 64, 639, 32, 0.0),     # the pre-pass took the last delta
    (BF, 3, 1001, 16, 64, 500, 33, 0.0),
    (BF, 1, 1200, 26, 64, 400, 0, 0.0),     # one unit: seven of eight do not exist
    (BF, 1, 700, 1, 64, 650, 130, 0.0),     # segments
    (FP, 1, 1003, 2, 128, 900, 5, 0.2),
    (BF, 1, 1024, 30, 128, 1000, 64, 0.0),  # rows of q and dO from global memory
    (BF, 1, 900, 1, 128, 899, 200, 0.0),
    (BF, 1, 1500, 20, 128, 512, 1, 0.0),
    # (the first two, and those of few deltas, take the kernel with two wavefronts per SIMD; the ones below this one, which
    # test_routes.py watches)
    (BF, 1, 2051, 20, 64, 512, 17, 0.0),
    (FP, 1, 1100, 26, 64, 1000, 6, 0.3),    # the last wavefront has one unit of two
    (FP, 4, 611, 20, 64, 2000, 33, 0.1),
    (BF, 1, 1003, 26, 128, 900, 40, 0.0),   # the pre-pass took the last delta
    (FP, 1, 2051, 20, 128, 900, 17, 0.2),
    (BF, 1, 2300, 40, 128, 1500, 1, 0.0),   # two units of four
    (BF, 1, 900, 8, 128, 899, 200, 0.0),    # segments
])
def test_kp_side_matches_the_fma_kernels(dtype, B, N, H, D, w1, w2, bias):
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(N + D)
    x = [torch.randn(B, N, H, D, generator=g, device="cuda").to(dtype) for _ in range(6)]
    kw = dict(k2_bias=bias, v2_bias=bias)
    out, lse = sa.simplicial_forward(*x[:5], w1, w2, **kw)
    needs = (True, False, True, False, True)
    got = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=needs, **kw)
    want = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=needs, flags=1, **kw)
    for name, i in (("dq", 0), ("dk2", 2), ("dv2", 4)):
        assert_close_rel(got[i], want[i].cpu(), 2e-2 if dtype == BF else 1.5e-2, name, atol=2e-3)
    again = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=(False, False, True, False, True), **kw)
    assert torch.equal(got[2], again[2]) and torch.equal(got[4], again[4])


@pytest.mark.parametrize("dtype,B,N,H,D,w1,w2,bias", [
    (BF, 1, 1100, 26, 128, 900, 24, 0.2),   # K' rows in fp32, with what the pre-pass left; q and dO rows in LDS
    (FP, 1, 1100, 26, 128, 900, 36, -0.2),  # ... the most deltas (37) that leave room for all three
    (BF, 1, 1100, 26, 128, 900, 38, 0.3),   # K' rows in 16 bits beside q and dO rows
    (FP, 1, 1024, 16, 128, 900, 57, 0.3),   # K' rows in fp32, q and dO rows from global memory
    (BF, 1, 1024, 16, 128, 900, 110, 0.1),  # neither
    (BF, 1, 1500, 30, 64, 500, 32, 0.2),    # two units
    (FP, 1, 1500, 30, 64, 500, 61, 0.2),
])
def test_k2_rows_in_both_forms(dtype, B, N, H, D, w1, w2, bias):
    """K' rows in LDS as (k2 + bias) * scale * log2(e) in fp32 or as they are, with a scale of its own: dQ, dK' and dV' as above."""
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(N + D + w2)
    x = [torch.randn(B, N, H, D, generator=g, device="cuda").to(dtype) for _ in range(6)]
    kw = dict(k2_bias=bias, v2_bias=-bias, scale=0.07)
    out, lse = sa.simplicial_forward(*x[:5], w1, w2, **kw)
    needs = (True, False, True, False, True)
    got = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=needs, **kw)
    want = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=needs, flags=1, **kw)
    for name, i in (("dq", 0), ("dk2", 2), ("dv2", 4)):
        assert_close_rel(got[i], want[i].cpu(), 2e-2 if dtype == BF else 1.5e-2, name, atol=2e-3)


@pytest.mark.parametrize("D,N,heads,w1,w2", [(64, 2051, 20, 513, 18), (128, 1003, 26, 901, 41)])
def test_layouts_and_half_open_windows(D, N, heads, w1, w2):
    """Views of one fused projection [B, N, 5, H, D] and of [B, H, N, D] tensors give what contiguous copies give, bit for bit, in all
    five gradients (the K-side kernel's too)."""
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(D)
    packed = torch.randn(1, N, 6, heads, D, generator=g, device="cuda").to(BF)
    x = packed.unbind(2)
    turned = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in x]
    plain = [t.contiguous() for t in x]
    kw = dict(window_inclusive=False)
    out, lse = sa.simplicial_forward(*plain[:5], w1, w2, **kw)
    want = sa.simplicial_backward(*plain[:5], out, lse, plain[5], w1, w2, **kw)
    for views in (x, turned):
        got = sa.simplicial_backward(*views[:5], out, lse, views[5], w1, w2, **kw)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    exact = sa.simplicial_backward(*plain[:5], out, lse, plain[5], w1, w2, flags=1, **kw)
    for name, a, b in zip(("dq", "dk1", "dk2", "dv1", "dv2"), want, exact):
        assert_close_rel(a, b.cpu(), 2e-2, name, atol=2e-3)


@pytest.mark.parametrize("D,N,heads,w1,w2", [(64, 2051, 20, 512, 17), (128, 1003, 26, 900, 40)])
def test_widely_spread_logits(D, N, heads, w1, w2):
    """fp16, logits of standard deviation 8: off by 8 * 2^-12 / sqrt(3) = 1.1e-3 each (products q*k2 rounded to 16 bits), 5e-3 at most, as are the
    weights, of which few are large: three times that covers a gradient, which has two of them (dS = P * (dP - D))."""
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(N)
    x = [(torch.randn(1, N, heads, D, generator=g, device="cuda") * (2 if t < 3 else 1)).to(FP) for t in range(6)]
    out, lse = sa.simplicial_forward(*x[:5], w1, w2)
    got = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2)
    want = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, flags=1)
    for name, a, b in zip(("dq", "dk1", "dk2", "dv1", "dv2"), got, want):
        assert_close_rel(a, b.cpu(), 1.5e-2, name, atol=2e-3)


@pytest.mark.parametrize("D,N,heads,w1,w2", [(64, 2051, 20, 512, 17), (128, 1003, 26, 900, 40)])
def test_a_gradient_that_is_not_a_number_stays_in_its_windows(D, N, heads, w1, w2):
    """Query r reaches its own row of dQ, its K' window of dK' and dV' and its K window of dK and dV (there to whole tiles of 32
    rows); everything else keeps its bits."""
    import simplical_attn_amd as sa
    r = N // 2
    g = torch.Generator(device="cuda").manual_seed(D)
    x = [torch.randn(1, N, heads, D, generator=g, device="cuda").to(BF) for _ in range(6)]
    out, lse = sa.simplicial_forward(*x[:5], w1, w2)
    clean = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2)
    x[5][:, r] = float("nan")
    got = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2)
    for a, b, lo, hi in zip(got, clean, (r, max(r - w1, 0) // 32 * 32, r - w2, max(r - w1, 0) // 32 * 32, r - w2), (r, r // 32 * 32 + 31, r, r // 32 * 32 + 31, r)):
        assert a[:, max(r - (w2 if hi == r and lo != r else 0), lo):r + 1].isnan().all()
        assert torch.equal(a[:, :lo], b[:, :lo]) and torch.equal(a[:, hi + 1:], b[:, hi + 1:])


@pytest.mark.parametrize("dtype,B,N,H,D,w1,w2,bias", [
    (BF, 1, 353, 8, 64, 2000, 130, 0.1),    # a sequence shorter than its window; segments
    (FP, 2, 513, 4, 64, 250, 32, 0.0),
    (BF, 1, 1111, 6, 64, 193, 6, -0.2),     # seven units of eight, the fewest deltas here
    (FP, 1, 1027, 27, 64, 160, 63, 0.3),
    (BF, 1, 1601, 17, 128, 233, 15, 0.1),
    (FP, 1, 1000, 40, 128, 260, 47, -0.3),
])
def test_narrower_windows_of_many_deltas(dtype, B, N, H, D, w1, w2, bias):
    """K windows of a few tiles, whose sweeps mostly begin and end inside one: dQ, dK' and dV' as above."""
    test_kp_side_matches_the_fma_kernels(dtype, B, N, H, D, w1, w2, bias)


def test_first_queries_do_not_depend_on_the_kernel():
    """dQ and dK' of the first queries, few large weights each, from this kernel (26 heads) and from the two-wavefront one (one of them): both round
    the weights there, so single elements differ by a flipped rounding of dS here and there, not by the weights' own (0.3 to 0.5 of the root mean
    square at w 1024/64; 0.01 here as it is)."""
    import simplical_attn_amd as sa
    from tests.test_routes import kp_route
    N, D, w1, w2 = 1003, 128, 900, 40
    assert kp_route(1, N, 26, D, w1, w2)[1] and not kp_route(1, N, 1, D, w1, w2)[1]
    g = torch.Generator(device="cuda").manual_seed(7)
    x = [(torch.randn(1, N, 26, D, generator=g, device="cuda") * s).to(BF) for s in (0.5, 0.5, 0.5, 1, 1, 1)]
    out, lse = sa.simplicial_forward(*x[:5], w1, w2)
    many = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=(True, False, True, False, True))
    for head in (0, 11, 25):
        y = [t[:, :, head:head + 1].contiguous() for t in (*x, out)]
        one = sa.simplicial_backward(*y[:5], y[6], lse[:, head:head + 1].contiguous(), y[5], w1, w2, needs=(True, False, True, False, True))
        for name, i in (("dq", 0), ("dk2", 2)):
            a, b = many[i][:, :, head:head + 1].float(), one[i].float()
            far = ((a - b).abs() / b.abs().clamp_min(b.pow(2).mean().sqrt().item()))[:, :16].max().item()
            assert far < 0.1, (name, head, far)
