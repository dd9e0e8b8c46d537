"""Dense patterns through every form of their reads, forward (P.V) and
backward (dV = P^T dO): the activation dtype with 16-byte rows, fp32 with
16-byte rows, and other storage types, strides and odd row pitches, at the
edges of the kernels' 64-query, 128-key and 256-query blocks and for batches
that do and do not share a pattern's workgroup.  Cells above the diagonal,
rows and columns past T and row padding hold NaN: none may be used.

The pattern is rounded to the activation dtype before the product, so the
reference is the float64 product of the rounded pattern and the rounded
inputs; what is left is fp32 accumulation and one output rounding (relative
2^-8 for bf16, 2^-11 for fp16; 1.5x that in relative L2)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pattern(P, S, T, layout, dtype, seed):
    """(P, S, S) device pattern of the layout, and its valid cells in float64."""
    g = torch.Generator().manual_seed(seed)
    p = torch.rand(P, S, S, generator=g).tril()
    p = p / p.sum(-1, keepdim=True)
    p = p.to(dtype)
    ref = p.double()
    keep = torch.ones(S, S, dtype=torch.bool).tril()
    keep[T:] = False
    nan = torch.full_like(p, float("nan"))
    p = torch.where(keep, p, nan).to(DEV)
    if layout == "padded":
        pitch = (S + 7) // 8 * 8 + 8
        buf = torch.full((P, S, pitch), float("nan"), device=DEV, dtype=dtype)
        buf[:, :, :S] = p
        p = buf[:, :, :S]
    elif layout == "transposed":
        p = p.transpose(1, 2).contiguous().transpose(1, 2)
    return p, ref[:, :T, :T]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("patt", ["same", "float32", "other"])
@pytest.mark.parametrize("layout", ["plain", "padded", "transposed"])
@pytest.mark.parametrize("T,S,B,hd", [(1, 8, 1, 64), (63, 64, 4, 64), (65, 101, 2, 64), (101, 101, 3, 128),
                                      (257, 257, 4, 64), (320, 336, 2, 128), (129, 136, 1, 96)])
def test_dense_pattern_forms(dtype, patt, layout, T, S, B, hd):
    import kernel
    pd = {"same": dtype, "float32": torch.float32,
          "other": torch.float16 if dtype == torch.bfloat16 else torch.bfloat16}[patt]
    P, ref = _pattern(3, S, T, layout, pd, seed=T + S)
    idx = [2, 0, 2]
    g = torch.Generator().manual_seed(T)
    v = torch.randn(B, 3, T, hd, generator=g).to(dtype)
    dy = torch.randn(B, 3, T, hd, generator=g).to(dtype)
    vd = v.to(DEV).requires_grad_()
    y = kernel.frozen_pv(P, vd, torch.tensor(idx, dtype=torch.int32, device=DEV), T)
    y.backward(dy.to(DEV))
    W = ref[idx].to(dtype).double()
    tol = 1.5 * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)
    for got, want, name in ((y, W @ v.double(), "y"), (vd.grad, W.transpose(1, 2) @ dy.double(), "dv")):
        got = got.detach().double().cpu()
        assert torch.isfinite(got).all(), name
        rel = float((got - want).norm() / want.norm())
        assert rel <= tol, f"{name}: rel {rel:.2e} > {tol:.2e}"


@pytest.mark.parametrize("patt", ["float32", "same"])
def test_dense_pattern_wide_pitch(patt):
    """Pattern rows 64 MB apart (one head's columns of a wide buffer): rows past
    the 2 GB that a buffer descriptor spans are read through pointers."""
    import kernel
    T = S = 48
    pitch = (64 << 20) // (4 if patt == "float32" else 2)
    pd = torch.float32 if patt == "float32" else torch.bfloat16
    P, ref = _pattern(1, S, T, "plain", pd, seed=3)
    wide = torch.empty(S * pitch, device=DEV, dtype=pd).as_strided((1, S, S), (S * pitch, pitch, 1))
    wide.copy_(P)
    g = torch.Generator().manual_seed(T)
    v, dy = (torch.randn(2, 2, T, 64, generator=g).bfloat16() for _ in range(2))
    vd = v.to(DEV).requires_grad_()
    y = kernel.frozen_pv(wide, vd, torch.zeros(2, dtype=torch.int32, device=DEV), T)
    y.backward(dy.to(DEV))
    W = ref.bfloat16().double()
    for got, want, name in ((y, W @ v.double(), "y"), (vd.grad, W.transpose(1, 2) @ dy.double(), "dv")):
        rel = float((got.detach().double().cpu() - want).norm() / want.norm())
        assert rel <= 1.5 * 2.0 ** -8, f"{name}: rel {rel:.2e}"
