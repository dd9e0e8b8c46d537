"""Tensors whose rows are closer than the head dimension: expanded over the
sequence (row stride 0), overlapping windows, and one row with a stride of
another layout.  The operator, its backward, frozen_pv and the pattern
gradients give what they give for the same values laid out contiguously, bit
for bit (the pattern gradients' sums are atomic: 1e-5 relative).  At the C entry
the float32 kernels read such rows; the 16-bit ones refuse them."""
import pytest
import torch

from saf_cases import closed_params, make_decomp, make_pattern, routing

pytestmark = pytest.mark.gpu
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _close_rows(shape, layout, dtype, seed):
    """A (B, N, T, hd) tensor of the layout."""
    B, N, T, hd = shape
    g = torch.Generator().manual_seed(seed)
    if layout == "expanded":
        return torch.randn(B, N, 1, hd, generator=g).to(dtype).to(DEV).expand(shape)
    if layout == "overlapping":
        step = 16
        x = torch.randn(B, N, step * (T - 1) + hd, generator=g).to(dtype).to(DEV)
        return x.unfold(2, hd, step)
    return torch.randn(B, N, hd, T, generator=g).to(dtype).to(DEV).transpose(2, 3)  # T = 1: row stride 1


def _call(T, hd, closed):
    """Routing and pattern arguments of five heads: two live, one dense, one
    decomposed, one closed form."""
    import kernel
    H, S = 5, (T + 63) // 64 * 64
    frozen, hidx, live = routing(H, {1: 1, 2: 2, 4: 2})
    alpha, rho, z = make_decomp(H, S, seed=T)
    ca, cr, cz = closed_params(H, S, {4: ("window", 9)})
    for t, c in zip((alpha, rho, z), (ca, cr, cz)):
        t[4] = c[4]
    cf = kernel.classify_closed_form(alpha, rho, z) if closed else None
    patt = make_pattern(H, S, seed=T + 1).to(DEV)
    kw = dict(alpha=alpha.to(DEV), rho=rho.to(DEV), z=z.to(DEV), closed_form=cf)
    return H, len(live), patt, frozen.to(DEV), hidx.to(DEV), kw


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("layout,T", [("expanded", 200), ("expanded", 33), ("overlapping", 200), ("one row", 1)])
@pytest.mark.parametrize("which", ["q", "k", "v"])
@pytest.mark.parametrize("hd", [64, 128])
def test_operator(dtype, layout, T, which, hd):
    import kernel
    H, U, patt, frozen, hidx, kw = _call(T, hd, closed=dtype != "fp32")
    B, dt = 2, DTYPES[dtype]
    base = {n: torch.randn(B, H if n == "v" else U, T, hd, generator=torch.Generator().manual_seed(i)).to(dt).to(DEV)
            for i, n in enumerate("qkv")}
    base[which] = _close_rows(base[which].shape, layout, dt, seed=T + hd)
    dy = torch.randn(B, H, T, hd, generator=torch.Generator().manual_seed(7)).to(dt).to(DEV)

    def run(t):
        t = {n: x.detach().requires_grad_() for n, x in t.items()}
        y = kernel.fused_mixed_attn(t["q"], t["k"], t["v"], patt, frozen, hidx, **kw)
        return (y, *torch.autograd.grad(y, (t["q"], t["k"], t["v"]), dy))

    got = run(base)
    want = run({n: x.clone(memory_format=torch.contiguous_format) for n, x in base.items()})
    for a, b, name in zip(got, want, ("y", "dq", "dk", "dv")):
        assert torch.equal(a, b), f"{name}: max difference {float((a.float() - b.float()).abs().max()):.2e}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T", [1, 70, 300])
def test_frozen_pv_sum(dtype, T):
    """The gradient of a sum over the sequence arrives with row stride 0, and
    with it dV = P^T 1."""
    import kernel
    dt = DTYPES[dtype]
    patt = make_pattern(3, T, seed=T).to(DEV)
    fz = torch.tensor([2, 0], dtype=torch.int32, device=DEV)
    v = torch.randn(2, 2, T, 64, generator=torch.Generator().manual_seed(T)).to(dt).to(DEV).requires_grad_()
    kernel.frozen_pv(patt, v, fz, T).sum(2).backward(torch.ones(2, 2, 64, device=DEV, dtype=dt))
    want = patt[[2, 0]].to(dt).double().sum(1)[None, :, :, None].expand(2, 2, T, 64)
    rel = float((v.grad.double() - want).norm() / want.norm())
    # one rounding of the result (2^-8 / 2^-11), or fp32 sums
    assert rel <= {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11, "fp32": 1e-6}[dtype], f"rel {rel:.2e}"


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_pattern_gradients_expanded(dtype):
    from supplement.trainable_pattern_kernels import pattern_gradients
    B, H, T, hd = 2, 3, 200, 64
    dt = DTYPES[dtype]
    alpha, rho, z = (t.to(DEV) for t in make_decomp(H, T, seed=3))
    g = torch.Generator().manual_seed(4)
    out, value = (torch.randn(B, H, T, hd, generator=g).to(dt).to(DEV) for _ in range(2))
    states = torch.tensor([2, 0, 2], dtype=torch.int32, device=DEV)
    grad = torch.randn(B, H, 1, hd, generator=g).to(dt).to(DEV).expand(B, H, T, hd)
    got = pattern_gradients(out, value, alpha, rho, z, states, grad)
    want = pattern_gradients(out, value, alpha, rho, z, states, grad.contiguous())
    for a, b in zip(got, want):
        assert float(b.norm()) > 0
        assert float((a - b).norm()) <= 1e-5 * float(b.norm())


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("which", ["k", "v"])
def test_library_entry(dtype, which, monkeypatch):
    """The C entry given the expanded tensor itself."""
    import kernel
    from kernel import fused_attn
    T, hd, B, dt = 100, 64, 2, DTYPES[dtype]
    H, U, patt, frozen, hidx, kw = _call(T, hd, closed=False)
    t = {n: torch.randn(B, H if n == "v" else U, T, hd, device=DEV).to(dt) for n in "qkv"}
    t[which] = _close_rows(t[which].shape, "expanded", dt, seed=1)
    call = lambda: kernel.fused_mixed_attn(t["q"], t["k"], t["v"], patt, frozen, hidx, **kw)
    want = call()
    monkeypatch.setattr(fused_attn, "_aligned_view", lambda x, align=16: x)
    if dtype == "fp32":
        assert torch.equal(call(), want)
    else:
        with pytest.raises(ValueError, match="closer than"):
            call()
