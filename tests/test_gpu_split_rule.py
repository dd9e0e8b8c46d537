"""Key-segment plans chosen by estimated time: live, dense and decomposed
heads at the shapes where the choice changes (first split, segment lengths of
8 to 32 blocks, back to unsplit with many heads; ragged last segments), and
the closed-form scan at one chunk and just past it, whose workspace is not
cleared by a launch.  Against the float64 oracle, at the bounds of the
operator's other forward tests (2e-2 max-abs, 1e-2 relative L2)."""
import pytest
import torch

from oracle import saf_oracle as orc
from saf_cases import closed_params, compare, f64, make_decomp, make_pattern, qkv, routing

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _dirty():
    """Leaves set bits in the allocator's free blocks, where the operator's
    workspace comes from."""
    for n in (1 << 10, 1 << 16, 1 << 20, 8 << 20):
        torch.full((n,), -1, device=DEV, dtype=torch.int32)


@pytest.mark.parametrize("kind", ["live", "dense16", "dense32", "decomp"])
@pytest.mark.parametrize("B,H,T,hd", [(1, 1, 577, 64), (1, 2, 1030, 64), (4, 6, 1030, 64), (1, 2, 2049, 64),
                                      (2, 6, 1999, 64), (1, 2, 1153, 128), (2, 3, 2047, 128), (1, 1, 1025, 32),
                                      (1, 1, 1025, 256)])
def test_segments(kind, B, H, T, hd):
    import kernel
    q, k, v = qkv(B, H, T, hd, seed=T + H, dtype=torch.bfloat16)
    state = {"live": 0, "dense16": 1, "dense32": 1, "decomp": 2}[kind]
    frozen, hidx, live = routing(H, {h: state for h in range(H)} if state else {})
    dev = lambda t: None if t is None else t.to(DEV)
    patt = pidx = None
    kw, okw = {}, {}
    if state == 1:
        patt = make_pattern(H, T + 8, seed=T).to(torch.bfloat16 if kind == "dense16" else torch.float32)
        pidx = torch.arange(H, dtype=torch.int32)
        okw = dict(pidx=pidx.numpy(), patt=f64(patt))
    elif state == 2:
        alpha, rho, z = make_decomp(H, T, seed=T)
        kw = dict(alpha=dev(alpha), rho=dev(rho), z=dev(z))
        okw = dict(alpha=f64(alpha), rho=f64(rho), z=f64(z))
    qd, kd = (q, k) if not state else (q[:, :0], k[:, :0])
    _dirty()
    y = kernel.fused_mixed_attn(dev(qd.contiguous()), dev(kd.contiguous()), dev(v), dev(patt), dev(frozen),
                                dev(hidx), dev(pidx), **kw)
    ref = orc.eager_mixed_attention(f64(q), f64(k), f64(v), frozen.numpy(), hidx.numpy(), **okw)
    compare(y, ref, what=f"{kind} B{B} H{H} T{T} hd{hd}")


@pytest.mark.parametrize("hd,chunk", [(32, 512), (64, 256), (96, 128), (128, 128), (256, 128)])
@pytest.mark.parametrize("dT", [None, -1, 0, 1])
def test_scan_of_one_chunk(hd, chunk, dT):
    import kernel
    B, H, T = 3, 3, 1 if dT is None else chunk + dT
    alpha, rho, z = closed_params(H, T, {0: ("mean", 0), 1: ("decay", 0.03), 2: ("window", 17)})
    cf = kernel.classify_closed_form(alpha, rho, z)
    _, _, v = qkv(B, H, T, hd, seed=T, dtype=torch.bfloat16)
    frozen = torch.full((H,), 2, dtype=torch.int32)
    none = torch.empty(B, 0, T, hd, device=DEV, dtype=torch.bfloat16)
    _dirty()
    y = kernel.fused_mixed_attn(none, none, v.to(DEV), None, frozen.to(DEV), alpha=alpha.to(DEV), rho=rho.to(DEV),
                                z=z.to(DEV), closed_form=cf, validate=True)
    ref = orc.eager_mixed_attention(f64(v), f64(v), f64(v), frozen.numpy(), alpha=f64(alpha), rho=f64(rho), z=f64(z))
    compare(y, ref, what=f"scan T{T} hd{hd}")
