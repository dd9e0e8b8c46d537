"""Calls that fork the library's second stream: the forward with decomposed
heads and a closed-form scan beside live ones, the backward with the frozen
heads' dV beside dQ and dK / dV (from an estimate of 170 us on: T >= 2900 at hd
64, T >= 1984 at hd 128), both also under graph capture.  Kernels give the same
rows whatever runs beside them, so joint calls equal separate ones bit for bit
(the scan's look-back order may move a last bit)."""
import pytest
import torch

from saf_cases import closed_params, make_decomp, make_pattern, qkv, routing

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _call(T, hd, dtype, states, closed=None, B=2):
    """Inputs of a call: q, k, v on the device, routing, patterns."""
    import kernel
    closed = closed or {}
    H, S = 1 + max([*states, *closed]), (T + 63) // 64 * 64
    frozen, hidx, live = routing(H, {**states, **{h: 2 for h in closed}})
    alpha, rho, z = make_decomp(H, S, seed=T, scale=0.6)
    for t, c in zip((alpha, rho, z), closed_params(H, S, closed)):
        for h in closed:
            t[h] = c[h]
    q, k, v = (t.to(DEV) for t in qkv(B, H, T, hd, seed=T + hd, dtype=dtype))
    patt = make_pattern(H, S, seed=3).to(DEV) if 1 in states.values() else None
    kw = dict(alpha=alpha.to(DEV), rho=rho.to(DEV), z=z.to(DEV), validate=False,
              closed_form=kernel.classify_closed_form(alpha, rho, z) if closed else None)
    return q, k, v, patt, frozen, hidx, live, kw


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("T,hd", [(3010, 64), (2049, 128)])
@pytest.mark.parametrize("kinds", [{1: 2, 3: 2, 4: 2}, {1: 1, 3: 1, 4: 1}, {1: 2, 3: 1, 4: 2}],
                         ids=["decomposed", "dense", "both"])
def test_forked_backward_equals_separate_calls(dtype, T, hd, kinds):
    """One call (which forks) against the live heads alone and each frozen head
    alone (which have nothing to fork)."""
    import kernel
    states = {0: 0, 2: 0, **kinds}
    q, k, v, patt, frozen, hidx, live, kw = _call(T, hd, dtype, states)
    H = len(states)
    dy = torch.randn(v.shape, generator=torch.Generator().manual_seed(5)).to(dtype).to(DEV)

    def grads(heads):
        lv = [h for h in heads if states[h] == 0]
        t = [x[:, lv].detach().requires_grad_() for x in (q, k)] + [v[:, heads].detach().requires_grad_()]
        fz = frozen[heads].to(DEV)
        hx = torch.tensor([lv.index(h) if h in lv else 0 for h in heads], dtype=torch.int32, device=DEV)
        px = torch.tensor(heads, dtype=torch.int32, device=DEV)
        sub = {n: x[heads] if torch.is_tensor(x) else x for n, x in kw.items()}
        y = kernel.fused_mixed_attn(*t, patt, fz, hx, px, **sub)
        g = torch.autograd.grad(y, [x for x in t if x.numel()], dy[:, heads])
        return (g[0], g[1], g[2]) if lv else (None, None, g[0])

    dq, dk, dv = grads(list(range(H)))
    for rep in range(2):   # a missing join shows when the next call reuses the memory
        again = grads(list(range(H)))
        assert all(torch.equal(a, b) for a, b in zip((dq, dk, dv), again))
    wq, wk, wv = grads(live)
    assert torch.equal(dq, wq) and torch.equal(dk, wk) and torch.equal(dv[:, live], wv)
    for h in kinds:
        assert torch.equal(dv[:, h:h + 1], grads([h])[2]), f"dv of head {h}"


@pytest.mark.parametrize("T,hd,forks", [(700, 64, False), (2100, 128, True)])
def test_default_forward_is_the_schedule_it_names(T, hd, forks):
    """decomp_unsplit None equals True where the library forks and False where
    it does not; the decomposed rows of the two agree to a bf16 step."""
    import kernel
    q, k, v, _, frozen, hidx, live, kw = _call(T, hd, torch.bfloat16, {0: 0, 1: 2, 2: 0, 3: 2, 4: 2})
    args = (q[:, live].contiguous(), k[:, live].contiguous(), v, None, frozen.to(DEV), hidx.to(DEV))
    y = {un: kernel.fused_mixed_attn(*args, decomp_unsplit=un, **kw) for un in (None, True, False)}
    assert torch.equal(y[None], y[forks])
    d = (y[True].float() - y[False].float()).abs()
    assert bool((d <= (y[False].float().abs() * 2.0 ** -7).clamp_min(2.0 ** -10)).all())


@pytest.mark.parametrize("backward", [False, pytest.param(True, marks=pytest.mark.skip(
    reason="the host process ended with a segmentation fault inside hipStreamEndCapture when a forked forward and its "
           "forked backward were captured together; the cause is not known, and a backward under capture no longer "
           "forks"))])
def test_forks_under_capture(backward):
    """Fork and join as graph edges: live, dense, decomposed and scan heads,
    replayed between eager calls on other inputs."""
    import kernel
    T, hd, dtype = 2100, 128, torch.bfloat16
    states = {0: 0, 1: 2, 2: 0, 3: 1, 4: 2, 5: 0}
    q, k, v, patt, frozen, hidx, live, kw = _call(T, hd, dtype, states, closed={6: ("decay", 0.03)})
    H = 7
    frozen, hidx = frozen.to(DEV), hidx.to(DEV)
    t = [x.contiguous().requires_grad_(backward) for x in (q[:, live], k[:, live], v)]
    dy = torch.randn(2, H, T, hd, generator=torch.Generator().manual_seed(5)).to(dtype).to(DEV)
    pidx = torch.arange(H, dtype=torch.int32, device=DEV)

    def run():
        y = kernel.fused_mixed_attn(*t, patt, frozen, hidx, pidx, decomp_unsplit=True, **kw)
        return (y, *torch.autograd.grad(y, t, dy)) if backward else (y,)

    want = [x.clone() for x in run()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            run()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for rep in range(3):
        other = run()
        for x in out:
            x.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            d = (a.float() - b.float()).abs()
            assert bool((d <= (b.float().abs() * 2.0 ** -7).clamp_min(2.0 ** -12)).all()), f"replay {rep}"
        assert torch.isfinite(other[0]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("layout", ["head-major view", "expanded over batch", "expanded over heads", "padded rows",
                                    "unaligned rows"])
@pytest.mark.parametrize("hd", [64, 128])
def test_gradient_layouts(dtype, layout, hd):
    """A gradient of any layout gives what its contiguous copy gives."""
    import kernel
    T = 300
    q, k, v, patt, frozen, hidx, live, kw = _call(T, hd, dtype, {0: 0, 1: 1, 2: 0, 3: 2, 4: 2})
    B, H = 2, 5
    t = [x.contiguous().requires_grad_() for x in (q[:, live], k[:, live], v)]
    g = torch.Generator().manual_seed(9)
    make = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)
    dy = {"head-major view": lambda: make(B, T, H, hd).transpose(1, 2),
          "expanded over batch": lambda: make(1, H, T, hd).expand(B, H, T, hd),
          "expanded over heads": lambda: make(B, 1, T, hd).expand(B, H, T, hd),
          "padded rows": lambda: make(B, H, T, hd + 8)[..., :hd],
          "unaligned rows": lambda: make(B, H, T, hd + 1)[..., 1:]}[layout]()
    pidx = torch.arange(H, dtype=torch.int32, device=DEV)
    y = kernel.fused_mixed_attn(*t, patt, frozen.to(DEV), hidx.to(DEV), pidx, **kw)
    got = torch.autograd.grad(y, t, dy)
    y = kernel.fused_mixed_attn(*t, patt, frozen.to(DEV), hidx.to(DEV), pidx, **kw)
    want = torch.autograd.grad(y, t, dy.contiguous())
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert torch.equal(a, b), name
