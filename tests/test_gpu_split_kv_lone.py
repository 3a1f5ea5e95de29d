"""dK and dV of the plane-split K side with one wavefront per SIMD where its stream of units can go wrong: one delta per query block, key blocks
that some or all wavefronts have no keys of, windows that begin and end in the middle of a block, more and fewer units than are formed
ahead, shares, both plane counts.  (fp16, few deltas of up to 80 queries: the kernel with two wavefronts per SIMD.)  Against the fp32 FMA kernels, to the bars of the other tests of these kernels (fp32 1e-5, 16 bits
half an ulp of the results and what D = sum dO * out loses with a rounded out: 2e-2, fp16 1e-2)."""
import pytest
import torch

from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu
BF, FP, F32 = torch.bfloat16, torch.float16, torch.float32
BAR = {BF: 2e-2, FP: 1e-2, F32: 1e-5}


@pytest.mark.parametrize("dtype,D", [(F32, 16), (F32, 32), (F32, 64), (BF, 40), (BF, 64 - 8), (BF, 72), (BF, 96), (FP, 48), (FP, 80)])
@pytest.mark.parametrize("B,N,H,w1,w2,bias", [
    (1, 1, 1, 0, 0, 0.0), (1, 33, 1, 0, 0, 0.0), (1, 300, 2, 40, 0, 0.1), (2, 129, 1, 128, 1, 0.0), (1, 97, 3, 31, 2, 0.0),
    (1, 200, 1, 500, 40, 0.2), (1, 161, 1, 3, 200, 0.0), (1, 700, 40, 129, 3, 0.0), (1, 520, 2, 95, 33, -0.1), (3, 40, 5, 40, 39, 0.0)])
def test_k_side_matches_the_fma_kernels(dtype, D, B, N, H, w1, w2, bias):
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(N + D)
    x = [torch.randn(B, N, H, D, generator=g, device="cuda").to(dtype) for _ in range(6)]
    kw = dict(k2_bias=bias, v2_bias=-bias)
    out, lse = sa.simplicial_forward(*x[:5], w1, w2, **kw)
    needs = (False, True, False, True, False)
    got = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=needs, **kw)
    want = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=needs, flags=1, **kw)
    for name, i in (("dk1", 1), ("dv1", 3)):
        # (a single triple per query: dK is rounding noise of size 2^-24 or, with a rounded out, 2^-9 of |dO||V||Q|)
        atol = (2e-5 if dtype == F32 else 0.2) if name == "dk1" and (w1 == 0 or N == 1) and w2 == 0 else 1e-6
        assert_close_rel(got[i], want[i].cpu(), BAR[dtype], name, atol=atol)
    again = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, needs=(False, False, False, True, False), **kw)
    assert torch.equal(got[3], again[3])
