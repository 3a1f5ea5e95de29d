"""dK and dV of the K-side kernel where its stream of units can go wrong: both numbers of K blocks per wavefront (grids of
64 .. 256 heads take two at head_dim 32 and 64), shares that begin inside a query block, blocks of one unit (w2 = 0), K'
windows that just fit LDS and that are walked in segments, first and last blocks cut by the windows.  Against the fp32 FMA
kernels on the same inputs; the products, weights and dS are rounded to 16 bits in between, which the bar of the other
16-bit tests (2e-2 of the largest element, fp16 1.5e-2) covers.  At 16 columns dP = sum of dout*v2 * v1 averages the roundings of its
products over a quarter of the terms that it has at 64, so its error may be sqrt(4) as large there (4e-2); 2.4e-2 is the largest
seen over five seeds, the same with the kernels whose P crosses between wavefronts in 16 bits, and 3e-2 the bar."""
import pytest
import torch

from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu
BF, FP = torch.bfloat16, torch.float16


@pytest.mark.parametrize("dtype,B,N,H,D,w1,w2,bias", [
    (BF, 4, 520, 64, 64, 300, 3, 0.0),      # two blocks per wavefront, not split
    (FP, 1, 400, 130, 64, 390, 0, 0.3),     # the same, a change of the query block behind every unit
    (BF, 1, 777, 256, 32, 500, 4, 0.0),
    (BF, 1, 300, 128, 16, 260, 9, 0.2),     # two blocks, shares, 16 columns
    (BF, 1, 257, 128, 32, 250, 200, 0.0),
    (BF, 1, 129, 1, 64, 40, 33, 0.0),       # one block, many shares
    (FP, 2, 33, 1, 128, 0, 1, 0.0),
    (BF, 1, 321, 1, 128, 31, 120, 0.0),     # the widest window that LDS holds ...
    (BF, 1, 321, 1, 128, 1000, 121, 0.0),   # ... and one more
    (BF, 1, 700, 1, 64, 33, 511, 0.1),
    (FP, 2, 17, 4, 64, 16, 16, 0.0),        # one query block, in shares of two and three units
    (BF, 1, 31, 2, 32, 20, 30, 0.2),
])
def test_k_side_matches_the_fma_kernels(dtype, B, N, H, D, w1, w2, bias):
    import simplical_attn_amd as sa
    g = torch.Generator(device="cuda").manual_seed(N + D)
    x = [torch.randn(B, N, H, D, generator=g, device="cuda").to(dtype) for _ in range(6)]
    kw = dict(k2_bias=bias, v2_bias=bias, needs=(False, True, False, True, False))
    out, lse = sa.simplicial_forward(*x[:5], w1, w2, k2_bias=bias, v2_bias=bias)
    got = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, **kw)
    want = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, flags=1, **kw)
    for name, i in (("dk1", 1), ("dv1", 3)):
        bar = 3e-2 if D == 16 else 2e-2 if dtype == BF else 1.5e-2
        assert_close_rel(got[i], want[i].cpu(), bar, name, atol=2e-3)
    again = sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, **kw)
    assert torch.equal(got[1], again[1]) and torch.equal(got[3], again[3])
