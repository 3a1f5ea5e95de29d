"""The head_dim 256 kernels at the sizes where their plans and rings turn: shares of the forward's rounds and its second
pass, segments of the K' window, shares of the K side, rings of rows that wrap several times, one-tile sweeps, biases and
strided rows; against the CPU oracle."""
import pytest
import torch

from simplical_attn_amd import _lib
from tests.util import assert_close_rel, make_inputs, oracle_all

pytestmark = pytest.mark.gpu
NAMES = ("out", "lse", "dq", "dk1", "dk2", "dv1", "dv2")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [(1, 140, 2, 60, 75, 0.0), (1, 33, 1, 8, 32, 0.2), (2, 64, 9, 31, 3, 0.0), (1, 300, 1, 290, 41, -0.3),
                                  (1, 32, 1, 31, 31, 0.0)])
def test_plans_rings_and_biases(dtype, case):
    import simplical_attn_amd as sa
    B, N, H, w1, w2, bias = case
    host = make_inputs(B, N, H, 256, seed=N + w2, dtype=dtype, mag=0.7)
    x = [t.cuda() for t in host]
    wide = [torch.stack([t, t], 3)[:, :, :, 0] for t in x]                     # the same rows with gaps between them
    want = dict(oracle_all(host, w1, w2, None, bias, bias))
    bar = 2e-2 if dtype == torch.bfloat16 else 1e-2
    got = []
    for inp in (x, wide):
        out, lse = sa.simplicial_forward(*inp[:5], w1, w2, None, bias, bias)
        grads = sa.simplicial_backward(*inp[:5], out, lse, inp[5], w1, w2, None, bias, bias)
        got.append(dict(zip(NAMES, (out, lse, *grads))))
    for name in NAMES:
        assert_close_rel(got[0][name], want[name], bar, name)
        assert torch.equal(got[0][name], got[1][name]), name
    only_k2 = sa.simplicial_backward(*x[:5], got[0]["out"], got[0]["lse"], x[5], w1, w2, None, bias, bias, needs=(False, False, True, False, False))
    assert torch.equal(only_k2[2], got[0]["dk2"])                              # (without dQ the rounds end without its sums)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,w2", [(96, 9), (96, 40), (700, 3)])
def test_weights_that_overflow_take_the_second_pass(dtype, N, w2):
    """Logits 0 on the latest keys, which fix the reference points, and 200 (288 octaves) on the earliest."""
    import simplical_attn_amd as sa
    q, k1, k2, v1, v2 = (torch.zeros(1, N, 1, 256) for _ in range(5))
    q[..., 0] = k2[..., 0] = 1.0
    k1[:, : N - 40, 0, 0] = 200.0 * 16
    g = torch.Generator().manual_seed(N)
    v1.normal_(generator=g)
    v2.normal_(generator=g)
    x = [t.to(dtype) for t in (q, k1, k2, v1, v2)]
    want = oracle_all([*x, x[0]], N, w2)
    out, lse = sa.simplicial_forward(*[t.cuda() for t in x], N, w2)
    assert_close_rel(out, want["out"], 2e-2 if dtype == torch.bfloat16 else 1e-2, "out")
    assert_close_rel(lse, want["lse"], 4e-3, "lse")                            # (the rounding of q * k2~ * scale, times 200)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("w2", [20, 21])
def test_a_query_that_is_not_a_number_stays_in_its_window(dtype, w2):
    """An even K' window has an odd number of deltas: the last round's second unit lies behind the window."""
    import simplical_attn_amd as sa
    x = [t.cuda() for t in make_inputs(1, 160, 1, 256, seed=3, dtype=dtype)]
    x[0][:, 50] = float("nan")
    out, lse = sa.simplicial_forward(*x[:5], 40, w2)
    dq, _, dk2, _, dv2 = sa.simplicial_backward(*x[:5], out, lse, x[5], 40, w2)
    rows = lambda t: t[0, :, 0].isnan().any(-1).nonzero()[:, 0].tolist()
    assert rows(dq) == [50] and rows(dk2) == rows(dv2) == list(range(50 - w2, 51))
