"""float32 kernels (attn_f32.hip) at the edges of their 32-row tiles and of the
four waves' block split, and through both forms of their pattern and LSE
reads, against the float64 oracle at the fp32 contract of test_gpu_f32.py
(forward max-abs 2e-5, gradients 2e-4)."""
import pytest
import torch

from oracle import saf_oracle as orc
from saf_cases import f64, make_decomp, make_pattern, routing, scale_of
from test_gpu_f32 import TOL_B, TOL_F, _maxabs, run_f32

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T", [1, 31, 32, 33, 97, 129, 161])
@pytest.mark.parametrize("hd", [64, 128, 256])
def test_f32_tile_edges(T, hd):
    # live, dense and decomposed heads; S > T leaves pattern columns past T
    run_f32(2, 5, T, hd, 192, [1], dec=[3], check_lse=True)


@pytest.mark.parametrize("layout", ["transposed_pattern", "padded_pattern", "strided_buffers", "strided_lse"])
def test_f32_pattern_and_lse_layouts(layout):
    """Pattern buffers that the 16-byte reads take (padded rows) and do not
    take (columns or buffers with a stride), and an LSE with a row stride."""
    import kernel
    B, H, T, hd, S = 2, 4, 100, 64, 128
    frozen, hidx, live = routing(H, {1: 1, 2: 2})
    patt = make_pattern(H, S, seed=5)
    alpha, rho, z = make_decomp(H, S, seed=6, scale=0.8)
    g = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn(B, H, T, hd, generator=g) for _ in range(3))
    dq, dk, dv = (t.to(DEV).requires_grad_() for t in (q[:, live].contiguous(), k[:, live].contiguous(), v))
    dpatt = patt.to(DEV)
    if layout == "transposed_pattern":
        dpatt = dpatt.transpose(1, 2).contiguous().transpose(1, 2)
    elif layout == "padded_pattern":
        pad = torch.full((H, S, S + 64), float("nan"), device=DEV)
        pad[:, :, :S] = dpatt
        dpatt = pad[:, :, :S]
    bufs = [t.to(DEV) for t in (alpha, rho, z)]
    if layout == "strided_buffers":
        bufs = [torch.stack([t, torch.full_like(t, float("nan"))], -1)[..., 0] for t in bufs]
    lse = torch.empty(B, T, H, device=DEV).transpose(1, 2) if layout == "strided_lse" else None
    y = kernel.fused_mixed_attn(dq, dk, dv, dpatt, frozen.to(DEV), hidx.to(DEV), alpha=bufs[0], rho=bufs[1], z=bufs[2],
                                lse=lse)
    kw = dict(patt=f64(patt), alpha=f64(alpha), rho=f64(rho), z=f64(z), sm_scale=scale_of(hd))
    args = (f64(q[:, live]), f64(k[:, live]), f64(v), frozen.numpy())
    _maxabs(y, orc.eager_mixed_attention(*args, hidx.numpy(), None, None, **kw), TOL_F, layout)
    w = torch.randn(y.shape, generator=g)
    (y * w.to(DEV)).sum().backward()
    refs = orc.eager_mixed_attention_grads(*args, f64(w), hidx.numpy(), None, **kw)
    for t, ref, name in zip((dq, dk, dv), refs, ("dq", "dk", "dv")):
        _maxabs(t.grad, ref, TOL_B, f"{name} {layout}")
