"""Row normalisers and their gradients at the edges of the kernels' 256-row
blocks, 2048-key chunks and 4-key steps, in the product form and where blocks
fall back to the direct one, against the float64 oracle.

z: each row sums at most S positive fp32 products in two levels, well under
1e-5 relative, so |dz| <= 1e-5 (1 + |z|) covers the sum, the fp32 exponent
arguments and the result's rounding.  Gradients: the terms' exponents carry
the rounding of values up to |z| (2^-23 |x| each), the sums run over S signed
terms: 1e-5 in relative L2."""
import numpy as np
import pytest
import torch

from oracle import saf_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(kind, H, S):
    g = torch.Generator().manual_seed(S + H)
    a = 0.5 * torch.randn(H, S, generator=g)
    r = -0.7 * torch.log1p(torch.arange(S, dtype=torch.float32)) + 0.2 * torch.randn(H, S, generator=g)
    if kind == "decay":     # distances far apart in exponent
        a = torch.zeros(H, S)
        r = -0.1 * torch.arange(S, dtype=torch.float32).repeat(H, 1)
    elif kind == "window":  # exact zeros and whole -inf chunks
        r = torch.where(torch.arange(S) < 70, r, torch.tensor(float("-inf")))
    elif kind == "spike":   # a key far above the rest: rows before it lie below its chunk's scale
        a[:, S // 2] = 120.0
    elif kind == "wide":    # logits of scale 40: past the product form's range
        a, r = 80 * a, 40 * torch.randn(H, S, generator=g)
    elif kind == "scale20":  # logits of scale 20: rows 2^-80 to 2^-132 below their chunk's scale
        a, r = 40 * a, 20 * r
    elif kind == "late":    # the first keys absent: rows without any key
        a[:, : min(S - 1, 130)] = float("-inf")
    return a, r


@pytest.mark.parametrize("kind", ["learned", "decay", "window", "spike", "wide", "scale20", "late"])
@pytest.mark.parametrize("S", [1, 5, 255, 256, 257, 2047, 2050, 2305, 4099])
def test_logz_blocks(kind, S):
    import kernel
    H = 2
    a, r = _inputs(kind, H, S)
    gz = torch.randn(H, S, generator=torch.Generator().manual_seed(1))
    ad, rd = a.to(DEV).requires_grad_(), r.to(DEV).requires_grad_()
    z = kernel.decomp_log_normalizers(ad, rd)
    ref = orc.decomposed_logz(a.double().numpy(), r.double().numpy())
    zh = z.detach().double().cpu().numpy()
    fin = np.isfinite(ref)
    assert np.array_equal(fin, np.isfinite(zh))
    assert (np.abs(zh - ref)[fin] <= 1e-5 * (1 + np.abs(ref[fin]))).all()
    da, dr = torch.autograd.grad(z, (ad, rd), gz.to(DEV))
    # the float64 gradients from the kernel's own z, as its backward takes it
    zz = torch.from_numpy(np.where(fin, zh, np.inf))
    wa, wr = torch.zeros(H, S, dtype=torch.float64), torch.zeros(H, S, dtype=torch.float64)
    for i in range(S):
        p = gz[:, i, None].double() * torch.exp(a[:, : i + 1].double() + r[:, : i + 1].double().flip(1) - zz[:, i, None])
        wa[:, : i + 1] += p
        wr[:, : i + 1] += p.flip(1)
    for got, want, name in ((da, wa, "dalpha"), (dr, wr, "drho")):
        got = got.double().cpu()
        assert torch.isfinite(got).all(), name
        err = float((got - want).norm()) / max(float(want.norm()), 1e-30)
        # exponent arguments of magnitude x round by 2^-23 |x|
        mag = float(torch.nan_to_num(a, neginf=0.0).abs().max() + torch.nan_to_num(r, neginf=0.0).abs().max())
        assert err <= 1e-5 + 2.0 ** -21 * mag, f"{name}: {err:.2e}"


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_gradient_of_one_row_not_finite(bad):
    """A gz_i that is not finite reaches the outputs o <= i and no other."""
    import kernel
    H, S, i = 1, 2305, 2060
    a, r = _inputs("learned", H, S)
    gz = torch.randn(H, S, generator=torch.Generator().manual_seed(1))
    grads = []
    for x in (0.0, bad):
        gz[0, i] = x
        ad, rd = a.to(DEV).requires_grad_(), r.to(DEV).requires_grad_()
        z = kernel.decomp_log_normalizers(ad, rd)
        grads.append(torch.autograd.grad(z, (ad, rd), gz.to(DEV)))
    for clean, got in zip(*grads):
        assert not torch.isfinite(got[0, : i + 1]).any()
        want, rest = clean[0, i + 1:], got[0, i + 1:]
        assert torch.isfinite(rest).all()
        # the two forms round their fp32 sums of a few hundred terms differently
        assert float((rest - want).norm()) <= 1e-5 * float(want.norm())


@pytest.mark.parametrize("exp", [-112, -104, 60, 115])
def test_gradient_scales_with_gz(exp):
    """gz times a power of two gives the gradients times that power, also where
    the logits' maxima lie far above every pair's value (a stripe's products
    then hold gz times up to 2^40 less than a pair is worth)."""
    import kernel
    H, S = 1, 700
    a, r = _inputs("learned", H, S)
    a[:, 300] += 13.5   # peaks that no row meets together: maxima 2^38 above any pair
    r[:, 500] += 13.5
    gz = torch.randn(H, S, generator=torch.Generator().manual_seed(2))
    grads = []
    for f in (1.0, 2.0 ** exp):
        ad, rd = a.to(DEV).requires_grad_(), r.to(DEV).requires_grad_()
        z = kernel.decomp_log_normalizers(ad, rd)
        grads.append(torch.autograd.grad(z, (ad, rd), (gz * f).to(DEV)))
    for one, got, name in zip(*grads, ("dalpha", "drho")):
        got = got.double() * 2.0 ** -exp
        # what 2^exp takes below the normal numbers is lost: 2^-126 / 2^exp
        err = (got - one.double()).abs()
        assert (err <= 1e-6 * one.double().abs() + 2.0 ** (-126 - exp)).all(), f"{name}: {float(err.max()):.2e}"


@pytest.mark.parametrize("which,lo,hi", [("alpha", 2048, 4096), ("alpha", 0, 2048), ("rho", 2000, 4500)])
def test_keys_not_a_number(which, lo, hi):
    """Rows that meet a NaN are NaN, also where a whole chunk of keys or of
    distances is; the others are what they are without it."""
    import kernel
    H, S = 1, 4500
    a, r = _inputs("learned", H, S)
    clean = kernel.decomposed_logz(a.to(DEV), r.to(DEV))
    (a if which == "alpha" else r)[:, lo:hi] = float("nan")
    z = kernel.decomposed_logz(a.to(DEV), r.to(DEV))
    assert torch.isnan(z[:, lo:]).all()
    # rows of the NaN's block take the direct form: fp32 rounding of z
    assert lo == 0 or float((z - clean)[:, :lo].abs().max()) <= 1e-5


@pytest.mark.parametrize("kind", ["learned", "window", "spike", "wide", "scale20", "late"])
@pytest.mark.parametrize("H,S", [(26, 2305), (32, 2048), (129, 257), (256, 255)])
def test_logz_rows_of_256(kind, H, S):
    """Calls with a work-group of 256 rows for every CU (the tests above have
    fewer and take 64) against each head alone."""
    import kernel
    a, r = (t.to(DEV) for t in _inputs(kind, H, S))
    z = kernel.decomposed_logz(a, r).double()
    for h in range(0, H, 1 if H < 100 else 17):
        one = kernel.decomposed_logz(a[h:h + 1].contiguous(), r[h:h + 1].contiguous())[0].double()
        fin = torch.isfinite(one)
        assert torch.equal(fin, torch.isfinite(z[h]))
        assert bool(((z[h] - one).abs()[fin] <= 1e-5 * (1 + one.abs()[fin])).all()), f"head {h}"

