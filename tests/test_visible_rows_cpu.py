"""Host side of the visible rows' autograd node: the differentiable form of its backward pass, on the CPU."""
import os
import sys
import types

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "citygs-x_amd"))

from gs_neural import _VisibleRows


@pytest.mark.parametrize("default_dtype", [torch.float32, torch.float64])
def test_differentiable_gradient_has_the_gradients_type(default_dtype):
    rank = torch.tensor([-1, 0, -1, 1], dtype=torch.int32)
    ctx = types.SimpleNamespace(saved_tensors=(rank,), needs_input_grad=(False, True, True, True, True, False), k=2)
    grads = [torch.randn(2, *s) for s in ((3,), (32,), (2, 3), (6,))] + [None]
    before = torch.get_default_dtype()
    torch.set_default_dtype(default_dtype)
    try:
        out = _VisibleRows.backward(ctx, *grads)  # (gradients are recorded: the form with a graph of its own)
    finally:
        torch.set_default_dtype(before)
    for d, g in zip(out[1:5], grads):
        assert d.dtype == torch.float32 and torch.equal(d[[1, 3]], g) and not d[[0, 2]].any()
