"""The native dispatcher kernels (csrc/torch_binding.cpp) without a GPU: fake device tensors go through the autograd kernel and end
in the Meta implementation, so what is accepted and what is refused can be checked here."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

import ops_rec


def attend(delta, **grads):
    """``hstu_jagged`` on fake device tensors, those named in ``grads`` requiring a gradient."""
    with FakeTensorMode():
        make = lambda name, *shape: torch.empty(*shape, dtype=torch.bfloat16, device="cuda", requires_grad=grads.get(name, False))  # noqa: E731
        q, k, v, mask = make("q", 7, 2, 64), make("k", 7, 2, 64), make("v", 7, 2, 64), make("mask", 2, 2, 8, 8)
        offs = torch.empty(3, dtype=torch.int32, device="cuda")
        args = (8, 8, 1.0, offs, offs) if delta else (8, 1.0, offs)
        return ops_rec.ascendc.attention.hstu_jagged(q, k, v, mask, None, 3, *args)


@pytest.mark.parametrize("delta", [False, True], ids=["equal", "delta"])
def test_a_mask_that_requires_grad_is_refused_only_where_a_gradient_is_recorded(delta):
    with torch.no_grad():
        assert attend(delta, mask=True).shape == (7, 2, 64)
        assert attend(delta, mask=True, q=True).shape == (7, 2, 64)
    for grads in (dict(mask=True), dict(mask=True, q=True)):
        with pytest.raises(NotImplementedError, match="mask is a non-differentiable input"):
            attend(delta, **grads)
    assert attend(delta, q=True).requires_grad and not attend(delta).requires_grad
