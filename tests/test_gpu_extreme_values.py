"""Values that the plane-split kernels (fp32 tensors, and 16-bit tensors of head dims without kernels of their own) do not
carry as sums of bf16 planes: infinities, NaN in rows that the windows leave out, fp32's lowest values as masks, and tensors
so small that their last plane is lost.  All must come out as on the fp32 FMA kernels, which sum valid pairs only."""
import pytest
import torch

from tests.util import make_inputs

pytestmark = pytest.mark.gpu
AUTO, GENERIC = 0, 1
BAR = {torch.float32: 3e-6, torch.float16: 2e-3, torch.bfloat16: 1.5e-2}      # relative 2-norm, two roundings apart
LAYOUTS = [(torch.float32, 64, 20), (torch.float32, 64, 3), (torch.float32, 128, 40), (torch.float32, 96, 20), (torch.float32, 16, 3),
           (torch.bfloat16, 96, 40), (torch.float16, 80, 3)]                  # few and many deltas: whole blocks and shares


def _inputs(dtype, D, what):
    x = [t.cuda() for t in make_inputs(1, 200, 2, D, seed=D, dtype=dtype)]
    inf, nan = float("inf"), float("nan")
    if what == "infinity in a value":
        x[4] = x[4].abs()
        x[3][:, 90, :, 5] = inf
    elif what == "minus infinity in a key":
        x[0], x[2] = x[0].abs(), x[2].abs()
        x[1][:, 90] = -inf
    elif what == "NaN value":
        x[3][:, 90] = nan
    elif what == "NaN query":
        x[0][:, 90, :, 1] = nan
    elif what == "NaN in every query":
        x[0][:, :, :, 2] = nan
    elif what == "nothing but NaN in the gradient":
        x[5][:] = nan
    elif what == "NaN in the queries of one head":
        x[0][:, :, 0, 2] = nan
    elif what == "infinity in V'":
        x[4][:, 90, :, 0] = inf
    elif what == "mask":
        x[0], x[2] = x[0].abs(), x[2].abs()
        x[1][:, 80:90] = torch.finfo(dtype).min
    elif what == "small values":
        x[3] = x[3] * 1e-36
    elif what == "NaN gradient":
        x[5][:, 90] = nan
    elif what == "small gradient":
        x[5] = x[5] * 1e-36
    elif what == "product above the range":
        x[4][:, 90], x[5][:, 95] = 1e30, 1e30
    elif what == "small keys":
        x[1] = x[1] * 1e-36
    return x


def _same(got, want, bar, name):
    got, want = got.double(), want.double()
    assert torch.equal(got.isnan(), want.isnan()), name
    assert torch.equal(got.isinf(), want.isinf()), name
    assert torch.equal(got[want.isinf()] > 0, want[want.isinf()] > 0), name
    ok = want.isfinite()
    diff, size = (got[ok] - want[ok]).norm().item(), want[ok].norm().item()
    assert diff <= bar * size, (name, diff, size)


FORWARD = ["NaN in every query", "NaN in the queries of one head", "infinity in a value", "minus infinity in a key", "NaN value", "NaN query", "infinity in V'", "mask", "small values", "small keys"]


def _cases(kinds):         # (the small tensors are an fp32 range)
    return [(*layout, what) for layout in LAYOUTS for what in kinds if layout[0] == torch.float32 or not what.startswith("small")]


@pytest.mark.parametrize("dtype,D,w2,what", _cases(FORWARD))
def test_forward(dtype, D, w2, what):
    import simplical_attn_amd as sa
    x = _inputs(dtype, D, what)
    got, want = (sa.simplicial_forward(*x[:5], 40, w2, flags=flags) for flags in (AUTO, GENERIC))
    _same(got[0], want[0], BAR[dtype], "out")
    _same(got[1], want[1], 1e-6, "lse")


BACKWARD = FORWARD + ["nothing but NaN in the gradient", "NaN gradient", "small gradient"]


@pytest.mark.parametrize("dtype,D,w2,what", _cases(BACKWARD) + [(torch.float32, 64, 20, "product above the range")])
def test_backward(dtype, D, w2, what):
    import simplical_attn_amd as sa
    x = _inputs(dtype, D, what)
    out, lse = sa.simplicial_forward(*x[:5], 40, w2, flags=GENERIC)
    got, want = (sa.simplicial_backward(*x[:5], out, lse, x[5], 40, w2, flags=flags) for flags in (AUTO, GENERIC))
    for name, a, b in zip(("dq", "dk1", "dk2", "dv1", "dv2"), got, want):
        _same(a, b, BAR[dtype], name)


def test_backward_of_a_subset_of_the_gradients():
    """The repaired launch writes what was asked for and nothing else."""
    import simplical_attn_amd as sa
    x = _inputs(torch.float32, 64, "NaN value")
    out, lse = sa.simplicial_forward(*x[:5], 40, 20)
    full = sa.simplicial_backward(*x[:5], out, lse, x[5], 40, 20)
    for needs in ((True, False, False, False, True), (False, True, False, False, False)):
        part = sa.simplicial_backward(*x[:5], out, lse, x[5], 40, 20, needs=needs)
        for need, a, b in zip(needs, part, full):
            assert (a is None) == (not need)
            assert a is None or torch.equal(a.nan_to_num(), b.nan_to_num())


def test_captured_step_follows_its_inputs():
    """A step captured on usual values, replayed on others: the verdict is the device's, at every replay."""
    import simplical_attn_amd as sa
    static = _inputs(torch.float32, 64, "")

    def step(x):
        out, lse = sa.simplicial_forward(*x[:5], 40, 40)
        return (out, lse, *sa.simplicial_backward(*x[:5], out, lse, x[5], 40, 40))

    step(static)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step(static)
    for what in ("NaN value", "", "infinity in a value", ""):
        new = _inputs(torch.float32, 64, what)
        for s, n in zip(static, new):
            s.copy_(n)
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in captured]
        for a, b in zip(got, step(new)):
            assert torch.equal(a.nan_to_num(7.0, 8.0, 9.0), b.nan_to_num(7.0, 8.0, 9.0)), what
        assert torch.isfinite(got[2]).all() == (what == "")
