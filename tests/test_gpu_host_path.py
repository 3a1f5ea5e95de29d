"""The module's native host path against TwoSimplicialAttentionFunction (same kernels, autograd formula in Python): every
subset of inputs that need gradients, broadcast inputs and upstream gradients, no_grad, a side stream and threads."""
import threading
import warnings

import pytest
import torch

from tests.util import make_inputs

pytestmark = pytest.mark.gpu
W1, W2 = 40, 9


def _grads(call, x, dout, needs):
    leaves = [t.clone().requires_grad_(n) for t, n in zip(x, needs)]
    out = call(*leaves)
    out.backward(dout)
    return [out.detach()] + [t.grad for t in leaves]


def _both(sa, D):
    fn = lambda *t: sa.TwoSimplicialAttentionFunction.apply(*t, W1, W2, None, 0.1, -0.2)
    return sa.TwoSimplicialAttention(D, W1, W2, None, 0.1, -0.2), fn


@pytest.mark.parametrize("needs", [(True,) * 5, (True, False, False, False, False), (False, True, False, True, False),
                                   (False, False, True, False, False), (False, False, False, False, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gradients_of_input_subsets(needs, dtype):
    import simplical_attn_amd as sa
    *x, dout = [t.cuda() for t in make_inputs(2, 100, 2, 64, seed=3, dtype=dtype)]
    module, fn = _both(sa, 64)
    # a broadcast key (stride 0 over heads) and a broadcast upstream gradient are copied, not refused
    x[1] = x[1][:, :, :1].expand(-1, -1, 2, -1)
    for d in (dout, dout[:, :1].expand_as(dout)):
        for a, b in zip(_grads(module, x, d, needs), _grads(fn, x, d, needs)):
            assert (a is None) == (b is None)
            assert a is None or torch.equal(a, b)
    with torch.no_grad():
        out = module(*[t.clone().requires_grad_(True) for t in x])
    assert not out.requires_grad and torch.equal(out, fn(*x))


def test_side_streams_and_threads():
    import simplical_attn_amd as sa
    *x, dout = [t.cuda() for t in make_inputs(1, 300, 2, 128, seed=4, dtype=torch.bfloat16)]
    module, fn = _both(sa, 128)
    want = _grads(fn, x, dout, (True,) * 5)
    torch.cuda.synchronize()
    got = [None] * 4

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(5):
                got[k] = _grads(module, x, dout, (True,) * 5)
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in got:
        assert all(torch.equal(a, b) for a, b in zip(g, want))


def _raised(call):
    try:
        call()
    except Exception as e:          # noqa: BLE001 - the kind is what is compared
        return type(e)
    return None


@pytest.mark.parametrize("which", [0, 3])
@pytest.mark.parametrize("grad", [True, False])
def test_forward_mode_derivatives_are_refused_not_dropped(which, grad):
    """There is no forward-mode formula: the module raises for a dual tensor, as the autograd function does, also where
    no input requires grad."""
    import torch.autograd.forward_ad as fwd

    import simplical_attn_amd as sa
    x = [t.cuda() for t in make_inputs(1, 64, 1, 64, seed=5, with_dout=False)]
    module, fn = _both(sa, 64)
    with fwd.dual_level(), torch.set_grad_enabled(grad):
        duals = list(x)
        duals[which] = fwd.make_dual(x[which], torch.ones_like(x[which]))
        assert _raised(lambda: module(*duals)) is _raised(lambda: fn(*duals)) is NotImplementedError
    assert torch.equal(module(*x), fn(*x))


@pytest.mark.parametrize("grad", [True, False])
def test_traced_module_computes_on_new_inputs(grad):
    import simplical_attn_amd as sa
    x, y = ([t.cuda().requires_grad_(grad) for t in make_inputs(1, 96, 2, 64, seed=s, with_dout=False)] for s in (6, 7))
    module, fn = _both(sa, 64)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        traced = torch.jit.trace(module, x, check_trace=False)
    assert any(n.kind() == "prim::PythonOp" for n in traced.graph.nodes())
    assert torch.equal(traced(*y), fn(*y)) and torch.equal(traced(*x), fn(*x))


@pytest.mark.parametrize("transform", ["grad", "vmap", "jvp"])
def test_function_transforms_raise_as_the_autograd_function_does(transform):
    import simplical_attn_amd as sa
    x = [t.cuda() for t in make_inputs(2, 64, 1, 64, seed=8, with_dout=False)]
    module, fn = _both(sa, 64)

    def outcome(call):
        if transform == "grad":
            return _raised(lambda: torch.func.grad(lambda q: call(q, *x[1:]).sum())(x[0]))
        if transform == "jvp":
            return _raised(lambda: torch.func.jvp(lambda q: call(q, *x[1:]), (x[0],), (x[0],)))
        return _raised(lambda: torch.func.vmap(call)(*[t[:, None] for t in x]))

    assert outcome(module) is outcome(fn) is not None


def test_saved_tensor_hooks_see_what_the_backward_needs():
    import simplical_attn_amd as sa
    *x, dout = [t.cuda() for t in make_inputs(1, 100, 2, 64, seed=9, dtype=torch.bfloat16)]
    module, fn = _both(sa, 64)
    want = _grads(fn, x, dout, (True,) * 5)
    with torch.autograd.graph.save_on_cpu():
        got = _grads(module, x, dout, (True,) * 5)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
