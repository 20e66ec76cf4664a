"""What the attention operator refuses before it looks at devices: forward-mode derivatives and function transforms,
of which its results would carry no trace, and the one problem whose folded normalisation has no gradient; and that the
attention classes are autograd functions."""
import types

import pytest
import torch

from reproducing_fastmax_results_amd.attention_mechanisms.score_function import (FASTMultiHeadAttention_Function,
                                                                                 FastmaxNormAttention)

CALLS = [lambda q, k, v: FASTMultiHeadAttention_Function.apply(q, k, v), FastmaxNormAttention.apply]


@pytest.mark.parametrize("call", CALLS)
@pytest.mark.parametrize("which", [0, 1, 2])
def test_forward_mode_is_refused(call, which):
    x = [torch.randn(1, 2, 8, 32) for _ in range(3)]
    with torch.autograd.forward_ad.dual_level():
        x[which] = torch.autograd.forward_ad.make_dual(x[which], torch.ones_like(x[which]))
        with pytest.raises(RuntimeError, match="forward-mode"):
            call(*x)
        with torch.no_grad(), pytest.raises(RuntimeError, match="forward-mode"):
            call(*x)


@pytest.mark.parametrize("call", CALLS)
def test_function_transforms_are_refused(call):
    x = [torch.randn(3, 1, 2, 8, 32) for _ in range(3)]
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.func.vmap(call)(*x)
    with pytest.raises(RuntimeError, match="functorch transforms"):
        torch.func.grad(lambda q: call(q, x[1][0], x[2][0]).sum())(x[0][0])
    with pytest.raises(RuntimeError, match="CUDA|cuda|device|GPU"):     # afterwards a call gets as far as the device check
        call(*(t[0] for t in x))


@pytest.mark.parametrize("grad", [False, True])
def test_folded_normalisation_refuses_more_keys_than_queries_under_the_mask(grad):
    """Two sub-problems would share one Jacobian: refused, with or without gradients, and not answered with the gradients
    of the normalised tensors.  (Unmasked, such a call gets as far as the device check.)"""
    q, k, v = (torch.randn(1, 2, n, 32, requires_grad=grad) for n in (8, 12, 12))
    with pytest.raises(RuntimeError, match="more keys than queries"):
        FastmaxNormAttention.apply(q, k, v, True)
    with pytest.raises(RuntimeError, match="CUDA|cuda|device|GPU"):
        FastmaxNormAttention.apply(q, k, v, False)


@pytest.mark.parametrize("cls", [FASTMultiHeadAttention_Function, FastmaxNormAttention])
def test_the_attention_classes_are_autograd_functions(cls):
    assert issubclass(cls, torch.autograd.Function)
    x = torch.randn(1, 2, 8, 32)
    with pytest.raises(RuntimeError, match="CUDA|cuda|device|GPU"):
        cls.forward(types.SimpleNamespace(needs_input_grad=(True,) * 3), x, x, x)
