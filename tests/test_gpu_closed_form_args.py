"""Closed-form tables of another length than the heads are refused (the library
reads one entry per output head)."""
import pytest
import torch

import kernel


@pytest.mark.gpu
@pytest.mark.parametrize("n_kind,n_param", [(3, 4), (5, 4), (4, 3)])
def test_closed_form_length(n_kind, n_param):
    H, T, hd = 4, 64, 64
    x = torch.zeros(1, H, T, hd, device="cuda", dtype=torch.bfloat16)
    rows = torch.zeros(H, T, device="cuda")
    closed = (torch.ones(n_kind, dtype=torch.int32, device="cuda"), torch.zeros(n_param, device="cuda"))
    with pytest.raises(ValueError):
        kernel.fused_mixed_attn(x, x, x, None, torch.full((H,), 2, dtype=torch.int32, device="cuda"), alpha=rows,
                                rho=rows, z=rows, closed_form=closed)
