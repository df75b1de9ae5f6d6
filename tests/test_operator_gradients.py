"""What the torch operators' autograd registration answers for calls without a
backward formula (shape functions on the meta device, no GPU)."""
from __future__ import annotations

import pytest
import torch

from scope_amd import library


def _head_bwd(y, grads):
    K, M = 6, 8
    iprm, fprm = [M, K, 128, 1, 0, 1], [0.0] * len(library._FPRM)
    om = torch.empty(K, device="meta")
    return library.coeff_head_bwd(y, om, om, None, None, grads + [None] * (len(library._HEAD_NAMES) - len(grads)), None,
                                  torch.empty(6, device="meta"), iprm, fprm)


def test_tensors_of_a_list_argument_are_constants():
    """As under ``torch.library.custom_op``: only tensor arguments make the
    result part of the graph, tensors inside a list argument do not."""
    y = torch.empty((1, 2, 128, 41), device="meta")
    g = torch.empty((1, 2, 128, 6), device="meta", requires_grad=True)
    assert not _head_bwd(y, [g]).requires_grad
    assert _head_bwd(y.clone().requires_grad_(), [g]).requires_grad


def test_no_formula_is_an_error_in_backward():
    y = torch.empty((1, 2, 128, 41), device="meta", requires_grad=True)
    out = _head_bwd(y, [])
    with pytest.raises(RuntimeError, match="coeff_head_bwd"):
        out.sum().backward()
    with torch.no_grad():
        assert not _head_bwd(y, []).requires_grad
