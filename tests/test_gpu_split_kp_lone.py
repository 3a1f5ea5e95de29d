"""dQ, dK' and dV' of the plane-split K' side with one wavefront per SIMD where its rounds and its stream of tiles can go wrong: wavefronts
without a unit in the last round, sweeps shorter than the tiles that are requested ahead, windows that begin and end in the middle of a
tile, a last tile that the sequence does not fill, segments, q and dO rows that do not fit LDS, both plane counts.  (Small grids with short
sweeps: some types' kernel with two wavefronts per SIMD; tests/test_routes.py says which.)  Against the fp32 FMA
kernels, to the bars of the other tests of these kernels (fp32 1e-5, bf16 2e-2, fp16 1e-2)."""
import pytest
import torch

from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu
BF, FP, F32 = torch.bfloat16, torch.float16, torch.float32
BAR = {BF: 2e-2, FP: 1e-2, F32: 1e-5}


@pytest.mark.parametrize("dtype,D", [(F32, 16), (F32, 32), (F32, 64), (BF, 40), (BF, 56), (BF, 72), (BF, 96), (FP, 48), (FP, 80)])
@pytest.mark.parametrize("B,N,H,w1,w2,bias", [
    (1, 1, 1, 0, 0, 0.0), (1, 33, 1, 0, 0, 0.0), (1, 300, 2, 40, 0, 0.1), (2, 129, 1, 128, 1, 0.0), (1, 97, 3, 31, 2, 0.0),
    (1, 200, 1, 500, 40, 0.2), (1, 161, 1, 3, 200, 0.0), (1, 700, 40, 129, 3, 0.0), (1, 520, 2, 95, 33, -0.1), (3, 40, 5, 40, 39, 0.0),
    (1, 640, 16, 70, 400, 0.1)])
def test_kp_side_matches_the_fma_kernels(dtype, D, B, N, H, w1, w2, bias):
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(N + D)
    x = [torch.randn(B, N, H, D, generator=g, device="cuda").to(dtype) for _ in range(6)]
    kw = dict(k2_bias=bias, v2_bias=-bias)
    out, lse = sa.simplicial_forward(*x[:5], w1, w2, **kw)
    needs = (True, False, True, False, True)
    got = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=needs, **kw)
    want = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=needs, flags=1, **kw)
    for name, i in (("dq", 0), ("dk2", 2), ("dv2", 4)):
        # (a single triple per query: dQ and dK' are rounding noise of size 2^-24 or, with a rounded out, 2^-9 of |dO||V||K|)
        atol = (2e-5 if dtype == F32 else 0.2) if name != "dv2" and (w1 == 0 or N == 1) and w2 == 0 else 1e-6
        assert_close_rel(got[i], want[i].cpu(), BAR[dtype], name, atol=atol)
    again = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=(False, False, True, False, True), **kw)
    assert torch.equal(got[2], again[2]) and torch.equal(got[4], again[4])


@pytest.mark.parametrize("dtype,D", [(F32, 16), (F32, 32), (F32, 64), (BF, 40), (BF, 56), (BF, 72), (BF, 96), (FP, 48), (FP, 80)])
@pytest.mark.parametrize("B,N,H,w1,w2,bias", [
    (1, 1, 300, 0, 0, 0.0), (1, 33, 130, 0, 0, 0.0), (1, 65, 90, 64, 11, 0.1), (2, 40, 80, 40, 39, 0.0), (1, 97, 70, 31, 2, -0.2), (1, 130, 60, 5, 1, 0.0)])
def test_short_sequences_of_many_heads(dtype, D, B, N, H, w1, w2, bias):
    """One to five tiles, more rounds than are at once on the chip."""
    test_kp_side_matches_the_fma_kernels(dtype, D, B, N, H, w1, w2, bias)
