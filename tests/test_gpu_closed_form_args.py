"""A closed-form kind table of another length than the heads, or a shorter
parameter table, is refused (the library reads one entry of each per output head)."""
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


@pytest.mark.gpu
def test_closed_form_longer_parameters():
    """A parameter table that holds more than the heads is accepted."""
    H, T, hd = 4, 64, 64
    v = torch.randn(1, H, T, hd, device="cuda", dtype=torch.bfloat16)
    none = v[:, :0].contiguous()
    rows = torch.zeros(H, T, device="cuda")
    z = torch.log1p(torch.arange(T, device="cuda").float()).repeat(H, 1)
    frozen = torch.full((H,), 2, dtype=torch.int32, device="cuda")
    kinds = torch.ones(H, dtype=torch.int32, device="cuda")
    y = [kernel.fused_mixed_attn(none, none, v, None, frozen, alpha=rows, rho=rows, z=z,
                                 closed_form=(kinds, torch.zeros(n, device="cuda"))) for n in (H, H + 3)]
    assert torch.equal(*y)
