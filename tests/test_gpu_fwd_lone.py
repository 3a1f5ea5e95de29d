"""The forward kernel with two units per wavefront where its rounds, its rings and its sweep from the queries' own tile down can go wrong:
wavefronts with one unit or none in the last round, a sweep of one tile, sequences that do not fill their last tile or block, K
windows wider than the sequence, K' windows that go round the ring of rows, shares of the rounds, the pre-pass's unit, logits that
leave the first reference point behind.  Against the fp32 FMA kernels on the same inputs; the products q*k2 and the weights are
rounded to 16 bits in between (bars of the other 16-bit tests)."""
import pytest
import torch

from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu
BF, FP = torch.bfloat16, torch.float16


@pytest.mark.parametrize("dtype,B,N,H,D,w1,w2,bias", [
    (BF, 1, 1000, 9, 64, 200, 9, 0.0),
    (FP, 1, 5000, 16, 128, 333, 12, 0.1),
    (BF, 4, 33, 40, 64, 5000, 0, 0.0),      # a sweep of one tile and one of two; seven of eight units do not exist
    (FP, 9, 31, 30, 64, 16, 40, 0.2),
    (BF, 1, 4115, 10, 128, 1000, 31, 0.0),
    (BF, 1, 640, 40, 64, 639, 32, 0.0),     # the pre-pass took the last delta
    (FP, 1, 4001, 26, 128, 300, 16, 0.0),
    (BF, 2, 517, 2, 64, 255, 200, 0.3),     # rows of K' and V' three times round their ring; shares
    (FP, 1, 900, 50, 64, 256, 130, 0.0),
    (BF, 1, 2500, 12, 128, 256, 150, 0.2),
    (BF, 2, 512, 4, 64, 256, 256, 0.0),
    (FP, 1, 5000, 24, 128, 600, 12, 0.1),   # head_dim 128 where the sweeps are long enough for this kernel (FwdLoneCfg::FIRST_PAYS)
    (BF, 1, 4001, 26, 128, 300, 32, 0.0),   # and with the pre-pass's unit
])
def test_forward_matches_the_fma_kernels(dtype, B, N, H, D, w1, w2, bias):
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(N + D)
    x = [torch.randn(B, N, H, D, generator=g, device="cuda").to(dtype) for _ in range(5)]
    kw = dict(k2_bias=bias, v2_bias=bias)
    out, lse = sa.simplicial_forward(*x, w1, w2, **kw)
    want, want_lse = sa.simplicial_forward(*x, w1, w2, flags=1, **kw)
    assert_close_rel(out, want.float().cpu(), 2e-2 if dtype == BF else 4e-3, "out")
    assert_close_rel(lse, want_lse.cpu(), 2e-2 if dtype == BF else 4e-3, "lse")
    again = sa.simplicial_forward(*x, w1, w2, **kw)
    assert torch.equal(out, again[0]) and torch.equal(lse, again[1])


@pytest.mark.parametrize("dtype", [BF, FP])
@pytest.mark.parametrize("D,w2,heads", [(64, 5, 20), (64, 45, 2), (64, 16, 60), (128, 30, 200), (128, 16, 400)])
def test_logits_that_leave_the_reference_point_behind(dtype, D, w2, heads):
    """Logits fall along the sequence, from 300 or 60 to 0 within a window: an early key outweighs the queries' own tile by hundreds of octaves."""
    import simplical_attn_amd as sa
    N, w1 = 470, 300
    ramp = torch.linspace(300.0, 0.0, N)
    ramp[200:] *= 0.2
    half = torch.full((1, N, heads, D), 0.5, device="cuda", dtype=dtype)
    k1 = ramp[None, :, None, None].expand(1, N, heads, D).to(dtype).cuda()
    g = torch.Generator(device="cuda").manual_seed(D)
    v1, v2 = (torch.randn(1, N, heads, D, generator=g, device="cuda").to(dtype) for _ in range(2))
    out, lse = sa.simplicial_forward(half, k1, half, v1, v2, w1, w2, 1 / (0.25 * D))
    want, want_lse = sa.simplicial_forward(half, k1, half, v1, v2, w1, w2, 1 / (0.25 * D), flags=1)
    # 0.25 * scale * log2(e) is rounded to 16 bits once for all keys: the exponents of the weights that share a row (differences of
    # logits up to a few units) are off by 2^-9 (fp16 2^-12) of themselves, the logits by as much of 300
    assert torch.isfinite(out.float()).all()
    assert_close_rel(out, want.float().cpu(), 2e-2, "out")
    assert_close_rel(lse, want_lse.cpu(), 4e-3, "lse")


@pytest.mark.parametrize("B,N,H,D,w1,w2,bias", [
    (1, 1000, 9, 64, 200, 9, 0.0),
    (1, 4115, 10, 128, 1000, 31, 0.0),
    (1, 4001, 26, 128, 300, 32, 0.0),       # the pre-pass's unit is computed again
    (1, 4100, 128, 128, 40, 31, 0.2),       # no tile that needs no mask
    (1, 2500, 12, 128, 256, 150, 0.0),
    (2, 517, 2, 64, 255, 200, 0.0),         # shares of four rounds, of which the first pass gives up the last two
])
def test_second_pass_on_widely_spread_logits(B, N, H, D, w1, w2, bias):
    """fp16 weights overflow in most blocks.  Logits of standard deviation 8 are off by 8 * 2^-12 / sqrt(3) = 1.1e-3 each (products q*k2
    rounded to 16 bits), 5e-3 at most, and an output averages what its largest weights have of it."""
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(N)
    x = [(torch.randn(B, N, H, D, generator=g, device="cuda") * (2 if t < 3 else 1)).to(FP) for t in range(5)]
    kw = dict(k2_bias=bias, v2_bias=bias)
    out, lse = sa.simplicial_forward(*x, w1, w2, **kw)
    want, want_lse = sa.simplicial_forward(*x, w1, w2, flags=1, **kw)
    assert_close_rel(out, want.float().cpu(), 4e-3, "out")
    assert_close_rel(lse, want_lse.cpu(), 4e-3, "lse")


@pytest.mark.parametrize("D,heads,w2", [(64, 24, 20), (128, 400, 31)])
def test_a_key_that_is_not_a_number_stays_in_its_window(D, heads, w2):
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(D)
    x = [torch.randn(1, 600, heads, D, generator=g, device="cuda").to(BF) for _ in range(5)]
    x[1][:, 350] = float("nan")
    out, lse = sa.simplicial_forward(*x, 230, w2)
    rows = lse[0].isnan()
    assert rows[:, 350:581].all() and rows.sum().item() == 231 * heads and torch.equal(out[0].isnan().any(-1).T, rows)


@pytest.mark.parametrize("D,N,heads,w1,w2", [(64, 1500, 6, 200, 20), (128, 4100, 16, 300, 24)])
def test_layouts_and_half_open_windows(D, N, heads, w1, w2):
    """Views of one fused projection [B, N, 5, H, D] and of [B, H, N, D] tensors give what contiguous copies give, bit for bit."""
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(D)
    packed = torch.randn(1, N, 5, heads, D, generator=g, device="cuda").to(BF)
    x = packed.unbind(2)
    turned = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in x]
    kw = dict(window_inclusive=False)
    want = sa.simplicial_forward(*[t.contiguous() for t in x], w1, w2, **kw)
    for views in (x, turned):
        got = sa.simplicial_forward(*views, w1, w2, **kw)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    exact, lse = sa.simplicial_forward(*x, w1, w2, flags=1, **kw)
    assert_close_rel(want[0], exact.float().cpu(), 2e-2, "out")
    assert_close_rel(want[1], lse.cpu(), 2e-2, "lse")


# The same where this kernel runs at head_dim 128 (FwdLoneCfg::FIRST_PAYS), with and without the pre-pass, and in shares (test_routes.py holds
# them to it)
@pytest.mark.parametrize("dtype", [BF, FP])
@pytest.mark.parametrize("D,w2,heads", [(128, 30, 300), (128, 24, 400), (64, 130, 6)])
def test_logits_that_leave_the_reference_point_behind_in_long_sweeps_and_shares(dtype, D, w2, heads):
    test_logits_that_leave_the_reference_point_behind(dtype, D, w2, heads)


def test_layouts_and_half_open_windows_in_long_sweeps():
    test_layouts_and_half_open_windows(128, 4100, 32, 300, 24)
