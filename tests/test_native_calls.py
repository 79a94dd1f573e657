"""The native call path under autograd's other modes and with arguments of other types: what the Python op call takes or
refuses, the native one does too.  Meta tensors run the dispatcher and autograd without a GPU."""
import pytest
import torch
import torch.autograd.forward_ad as forward_ad

from self_attention import self_attention
from streaming_attention import streaming_attention


def _meta(requires_grad=False):
    return torch.randn(2, 3, 64, 32, device="meta", requires_grad=requires_grad)


def _call(q, **kw):
    return streaming_attention(q, _meta(), _meta(), None, 16, 2, **kw)


@pytest.mark.parametrize("requires_grad", [False, True])
def test_forward_mode_is_refused(requires_grad):
    with forward_ad.dual_level(), pytest.raises(NotImplementedError):
        _call(forward_ad.make_dual(_meta(requires_grad), _meta()))
    with pytest.raises(RuntimeError):
        torch.func.jvp(_call, (_meta(),), (_meta(),))


def test_undefined_output_gradient_counts_as_zero():
    class NoGrad(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x * 1

        @staticmethod
        def backward(ctx, g):
            return None

    q = _meta(True)
    grad, = torch.autograd.grad(NoGrad.apply(_call(q)).sum(), q, allow_unused=True)
    assert grad is not None and grad.shape == q.shape


@pytest.mark.parametrize("kw", [dict(sm_scale=torch.tensor(0.5)), dict(sm_scale=1), dict(autotune=1), dict(return_lse=1),
                                dict(prescale_qk=None)])
def test_convertible_arguments_are_taken(kw):
    out = _call(_meta(), **kw)
    assert (out[0] if kw.get("return_lse") else out).shape == (2, 3, 64, 32)


@pytest.mark.parametrize("kw", [dict(sm_scale="x"), dict(autotune="x"), dict(prescale_qk=[1]), dict(precision=None)])
def test_other_arguments_are_refused_by_the_op(kw):
    with pytest.raises(RuntimeError, match="Expected a value of type"):
        _call(_meta(), **kw)


def test_dense_is_forward_only():
    q = _meta(True)
    out = self_attention(q, _meta(), _meta(), None)
    assert out.requires_grad
    with pytest.raises(RuntimeError, match="no autograd formula"):
        torch.autograd.grad(out.sum(), q)


def test_backward_runs_under_compiled_autograd():
    from torch._dynamo import compiled_autograd

    q = _meta(True)
    out, lse = _call(q, return_lse=True)
    assert not lse.requires_grad and lse.grad_fn is None
    with compiled_autograd._enable(torch.compile(backend="eager")):
        out.sum().backward()
    assert q.grad.shape == q.shape
