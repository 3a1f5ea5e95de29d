"""bf16 tensors of the head dims in between: without biases a product q*k2 or dO*v2 has 16 bits, which two planes hold exactly, and the
kernels take two where a bias asks for three.  A bias of 1e-30 changes no value (k2 + 1e-30 = k2) but the path: both must be equally
far from the fp64 oracle.  What differs between them are fp32 roundings, 2^-15 of the rounding of the results, so that the errors differ by
results on a tie: 1 % is far above that."""
import pytest
import torch

from tests.util import make_inputs, oracle_all

pytestmark = pytest.mark.gpu
NAMES = ("out", "lse", "dq", "dk1", "dk2", "dv1", "dv2")


@pytest.mark.parametrize("D", [8, 40, 72, 80, 96, 104, 120])
@pytest.mark.parametrize("B,N,H,w1,w2,scale", [(1, 33, 1, 5, 1, None), (2, 97, 2, 33, 8, 0.3), (1, 160, 3, 40, 130, None), (1, 300, 1, 310, 0, 0.05), (1, 63, 2, 0, 31, 1.0)])
def test_two_planes_are_as_exact_as_three(D, B, N, H, w1, w2, scale):
    import simplical_attn_amd as sa
    host = make_inputs(B, N, H, D, seed=D + N, dtype=torch.bfloat16)
    want = oracle_all([x.double() for x in host], w1, w2, scale, 0.0, 0.0)
    x = [t.to("cuda:0") for t in host]
    error = {}
    for bias in (0.0, 1e-30):
        out, lse = sa.simplicial_forward(*x[:5], w1, w2, scale, bias, bias)
        got = (out, lse) + sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, scale, bias, bias)
        error[bias] = {n: (g.double().cpu() - want[n].double()).norm().item() for n, g in zip(NAMES, got)}
        size = {n: want[n].double().norm().item() for n in NAMES}
    for n in NAMES:
        assert error[0.0][n] <= 1.01 * error[1e-30][n] + 2e-5 * size[n], (n, error[0.0][n] / size[n], error[1e-30][n] / size[n])


@pytest.mark.parametrize("D", [8, 24, 72, 96, 104, 120])
@pytest.mark.parametrize("heads", [1, 40])
def test_a_scale_that_cannot_wait(D, heads):
    """q*k2 is no float here (2^-140), scale*q*k2 and the logits are: three planes with the scale in them, in every forward and in the backward."""
    import simplical_attn_amd as sa
    host = make_inputs(1, 63, heads, D, seed=D, dtype=torch.bfloat16)
    host[0], host[2], host[1] = host[0] * 2.0 ** -70, host[2] * 2.0 ** -70, host[1] * 2.0 ** 60
    scale = 2.0 ** 80 * D ** -0.5
    want = oracle_all([x.double() for x in host], 40, 9, scale)
    x = [t.to("cuda:0") for t in host]
    out, lse = sa.simplicial_forward(*x[:5], 40, 9, scale)
    got = (out, lse) + sa.simplicial_backward(*x[:5], out, lse, x[5], 40, 9, scale)
    assert want["lse"].std() > 0.5
    for n, g in zip(NAMES, got):
        error = (g.double().cpu() - want[n].double()).norm() / want[n].double().norm()
        assert error < (1e-6 if n == "lse" else 1e-2), (n, error)


@pytest.mark.parametrize("D", [40, 72, 96])
def test_logits_that_overflow_without_the_scale(D):
    """One key with a logit of 2^128 * scale, the largest of every row that sees it: P is 0 or 1 (all of these are powers of two, so that logit and LSE
    agree to the last bit), and dV and dV' are those of the fp32 FMA kernels."""
    import simplical_attn_amd as sa
    x = [t.cuda() for t in make_inputs(1, 150, 2, D, seed=D, dtype=torch.bfloat16)]
    x[0][..., 0], x[2][..., 0] = 2.0, 1.0
    x[1][:, 37, :, 0] = 2.0 ** 127
    out, lse = sa.simplicial_forward(*x[:5], 60, 9, 0.125)
    assert torch.isfinite(out).all() and lse.max() > 1e37
    got = sa.simplicial_backward(*x[:5], out, lse, x[5], 60, 9, 0.125)
    want = sa.simplicial_backward(*x[:5], out, lse, x[5], 60, 9, 0.125, flags=1)
    for t in (3, 4):
        assert (got[t] - want[t]).abs().max() <= 1e-2 * want[t].abs().max()
    assert all(torch.equal(a.isnan(), b.isnan()) for a, b in zip(got, want))
