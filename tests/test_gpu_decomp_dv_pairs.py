"""dV of decomposed heads with two sequences per workgroup (hd <= 64, an even
batch, three workgroups per CU before pairing) against the same sequences one
by one, which run unpaired: the arithmetic of a sequence does not depend on
its partner, so the gradients are equal bit for bit.  One step below the
rule's edge and an odd batch stay unpaired on both sides."""
import pytest
import torch

from saf_cases import make_decomp

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("B,F,T,hd", [(8, 11, 1100, 64), (6, 16, 1024, 64), (6, 16, 1023, 32), (8, 11, 1025, 32),
                                      (12, 11, 768, 64), (7, 16, 1024, 64)])
def test_pairs_equal_single_sequences(B, F, T, hd, dtype):
    import kernel
    H = F + 1
    g = torch.Generator().manual_seed(T + B)
    x = [torch.randn(B, n, T, hd, generator=g).to(dtype).to(DEV) for n in (1, 1, H, H)]
    alpha, rho, z = (t.to(DEV) for t in make_decomp(H, T, seed=T))
    frozen = torch.full((H,), 2, dtype=torch.int32, device=DEV)
    frozen[0] = 0
    hidx = torch.zeros(H, dtype=torch.int32, device=DEV)

    def dv(sl):
        q, k, v = (t[sl].detach().requires_grad_() for t in x[:3])
        y = kernel.fused_mixed_attn(q, k, v, None, frozen, hidx, alpha=alpha, rho=rho, z=z)
        return torch.autograd.grad(y, (q, k, v), x[3][sl])[2]

    got = dv(slice(0, B))
    assert torch.isfinite(got).all()
    for b in range(B):
        assert torch.equal(got[b:b + 1, 1:], dv(slice(b, b + 1))[:, 1:]), f"sequence {b}"
