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
