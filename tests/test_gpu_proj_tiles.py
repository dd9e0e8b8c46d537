"""Projection GEMMs: problems of many tiles (256 x 256) and of few (128 x 128)
run the same products in the same order, so a row's result must not depend on
how many rows come with it.  Ragged row counts on both sides of the choice."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op,hd", [("gelu", 0), ("swiglu", 0), ("rope", 64), ("rope", 128)])
@pytest.mark.parametrize("M", [1100, 1537])
def test_rows_do_not_depend_on_the_tile(op, hd, M):
    import kernel
    N, K = 8192, 256  # M rows: 160 and more big tiles; 1 to 511 rows: at most 64
    g = torch.Generator(device="cuda").manual_seed(M + hd)
    x = torch.randn(1, M, K, device="cuda", generator=g).bfloat16()
    w = (0.1 * torch.randn(N, K, device="cuda", generator=g)).bfloat16()
    cos, sin = (torch.randn(M, max(hd, 1), device="cuda", generator=g).bfloat16() for _ in range(2))

    def run(lo, hi):
        xs = x[:, lo:hi].contiguous()
        if op == "gelu":
            return kernel.linear_gelu(xs, w)
        if op == "swiglu":
            return kernel.linear_swiglu(xs, w)
        return kernel.linear_rope(xs, w, 4096, hd, cos[lo:hi].contiguous(), sin[lo:hi].contiguous())

    full = run(0, M)
    assert torch.isfinite(full).all()
    for lo, hi in ((0, 1), (3, 130), (255, 766), (M - 129, M)):
        assert torch.equal(run(lo, hi), full[:, lo:hi]), (lo, hi)
