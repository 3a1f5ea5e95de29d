"""Head dims between the kernels' own widths run in the next wider kernel (16-bit tensors other than head_dim 16: on the
plane-split kernels), whose columns from head_dim on read as zeros and are not written.  Against the CPU oracle, on views
into wider rows whose columns past head_dim hold NaN (a read past a row's end would poison the result), and on
contiguous tensors with the same bits."""
import pytest
import torch

from simplical_attn_amd import _lib
from tests.util import assert_close_rel, make_inputs, oracle_all

pytestmark = pytest.mark.gpu
NAMES = ("out", "lse", "dq", "dk1", "dk2", "dv1", "dv2")
BAR = {torch.bfloat16: 2e-2, torch.float16: 1e-2, torch.float32: 1e-5}


def _run(x, w1, w2, kb, vb):
    import simplical_attn_amd as sa
    out, lse = sa.simplicial_forward(*x[:5], w1, w2, None, kb, vb)
    return (out, lse) + sa.simplicial_backward(*x[:5], out, lse, x[5], w1, w2, None, kb, vb)


# (N, w1, w2): ragged tiles, the pre-pass multiples, K'/V' rows too many for LDS copies, a K' window in segments
@pytest.mark.parametrize("D", [8, 16, 40, 80, 96, 120])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(97, 33, 8), (160, 40, 130)], ids=lambda s: "N%d-w%d_%d" % s)
def test_head_dims_between_the_kernel_widths(D, dtype, shape):
    N, w1, w2 = shape
    B, H, kb, vb = 2, 2, 0.1, -0.2
    host = make_inputs(B, N, H, D, seed=D + N, dtype=dtype)
    dev = torch.device("cuda:0")
    wide = [torch.full((B, N, H, D + 8), float("nan"), dtype=dtype, device=dev) for _ in host]
    views = [w[..., :D] for w in wide]
    for v, x in zip(views, host):
        v.copy_(x)
    got = dict(zip(NAMES, _run(views, w1, w2, kb, vb)))
    want = oracle_all(host, w1, w2, None, kb, vb)
    for name in NAMES:
        assert_close_rel(got[name], want[name], BAR[dtype], name)
    for name, g in zip(NAMES, _run([x.to(dev) for x in host], w1, w2, kb, vb)):
        assert torch.equal(got[name], g), name


def test_pre_pass_kernels_at_a_width_between():
    """A grid large enough for the pre-pass of both directions (N / 32 * B * H >= 768, w2 a multiple of 8), head_dim 80
    and 16, against the fp32 FMA kernels."""
    import simplical_attn_amd as sa
    dev = torch.device("cuda:0")
    for D in (16, 80):
        x = [t.to(dev) for t in make_inputs(2, 1550, 8, D, seed=D, dtype=torch.bfloat16)]
        out, lse = sa.simplicial_forward(*x[:5], 40, 16)
        grads = sa.simplicial_backward(*x[:5], out, lse, x[5], 40, 16)
        f = _lib.FLAG_FORCE_GENERIC
        rout, rlse = sa.simplicial_forward(*x[:5], 40, 16, flags=f)
        rgrads = sa.simplicial_backward(*x[:5], rout, rlse, x[5], 40, 16, flags=f)
        for name, a, b in zip(NAMES, (out, lse, *grads), (rout, rlse, *rgrads)):
            assert_close_rel(a, b.float().cpu(), 2e-2, "%s D%d" % (name, D))
