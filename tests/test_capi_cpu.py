"""C-ABI checks that need no GPU: libsafattn.so loads, exports every entry
point declared in include/saf_attn.h, and rejects invalid arguments with a
status and message before any device work is enqueued."""
import ctypes
import os
import re

import pytest
import torch

from kernel import _ext

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(REPO, "include", "saf_attn.h")


def _declared():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"\b(saf_[a-z_0-9]+)\s*\(", text)))


def test_library_loads_and_exports_header_symbols():
    L = _ext.lib()
    declared = _declared()
    assert declared, "no declarations found"
    for name in declared:
        assert hasattr(L, name), f"{name} declared in saf_attn.h but not exported"
    assert set(declared) == set(_ext.EXPORTS)
    assert L.saf_version().startswith(b"saf-mi355x")


def test_workspace_bytes():
    L = _ext.lib()
    assert L.saf_workspace_bytes(8, 16384, 64, 0) == 0
    # 256-byte header (error word) + one 8-byte status word per (sequence,
    # 256-row chunk, column) at hd 64
    n = L.saf_workspace_bytes(8, 16384, 64, 12)
    nseq, nch = 8 * 12, 16384 // 256
    assert n == 256 + 8 * nseq * nch * 64
    assert L.saf_workspace_bytes(1, 1000, 128, 1) == 256 + 8 * 8 * 128   # 128-row chunks at hd 128
    assert L.saf_workspace_bytes(1, 1000, 80, 3) == 0   # unsupported head dim


def _args(H=4, T=64, hd=64, dtype=_ext.SAF_BF16, frozen=None, ptr=0x100000):
    a = _ext.SafMixedAttnArgs()

    def t4(shape):
        d = _ext.SafTensor()
        d.data, d.dtype, d.ndim = ptr, dtype, 4
        st = [shape[1] * shape[2] * shape[3], shape[2] * shape[3], shape[3], 1]
        for i in range(4):
            d.size[i], d.stride[i] = shape[i], st[i]
        return d

    a.q = t4((1, H, T, hd))
    a.k = t4((1, H, T, hd))
    a.v = t4((1, H, T, hd))
    a.out = t4((1, H, T, hd))
    a.n_heads = H
    fz = frozen if frozen is not None else [0] * H
    a._keep = (ctypes.c_int32 * H)(*fz)
    a.frozen = a._keep
    a.sm_scale = 0.125
    return a


@pytest.mark.parametrize("mutate,code,msg", [
    (lambda a: setattr(a, "n_heads", 0), _ext.SAF_EUNSUPPORTED, "n_heads"),
    (lambda a: setattr(a.v, "dtype", _ext.SAF_I32), _ext.SAF_EUNSUPPORTED, "int32"),
    (lambda a: setattr(a.v, "dtype", _ext.SAF_F32), _ext.SAF_EINVAL, "dtype must match"),
    (lambda a: a.v.size.__setitem__(3, 80), _ext.SAF_EUNSUPPORTED, "head_dim"),
    (lambda a: a.out.size.__setitem__(2, 63), _ext.SAF_EINVAL, "out must have shape"),
    (lambda a: a.v.stride.__setitem__(3, 2), _ext.SAF_EALIGN, "contiguous last"),
    (lambda a: setattr(a.v, "data", 0x100002), _ext.SAF_EALIGN, "aligned"),
    (lambda a: a._keep.__setitem__(0, 5), _ext.SAF_EINVAL, "head state"),
    (lambda a: a._keep.__setitem__(0, 1), _ext.SAF_EINVAL, "require patt"),
    (lambda a: setattr(a, "frozen", None), _ext.SAF_EINVAL, "frozen"),
])
def test_invalid_arguments_rejected_without_launch(mutate, code, msg):
    L = _ext.lib()
    a = _args()
    mutate(a)
    rc = L.saf_mixed_attn_fwd(ctypes.byref(a), None)
    assert rc == code
    assert msg in L.saf_last_error().decode()


def test_closed_form_needs_workspace():
    L = _ext.lib()
    a = _args(frozen=[0, 2, 0, 0])
    kinds = (ctypes.c_int32 * 4)(0, 1, 0, 0)
    prm = (ctypes.c_float * 4)(0, 0, 0, 0)
    a.closed_kind, a.closed_param = kinds, prm
    rc = L.saf_mixed_attn_fwd(ctypes.byref(a), None)
    assert rc == _ext.SAF_EWORKSPACE
    kinds[1] = 2
    prm[1] = -1.0
    assert L.saf_mixed_attn_fwd(ctypes.byref(a), None) == _ext.SAF_EINVAL
    assert "decay rate" in L.saf_last_error().decode()


def test_cpu_tensors_fail_loudly():
    import kernel
    q = torch.zeros(1, 1, 4, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="HIP devices only"):
        kernel.fused_mixed_attn(q, q, q, None, torch.zeros(1, dtype=torch.int32))
    with pytest.raises(RuntimeError, match="HIP devices only"):
        kernel.frozen_pv(torch.zeros(1, 4, 4), q, torch.zeros(1, dtype=torch.int32), 4)


def test_host_table_cached_per_tensor_and_version():
    """The routing tables are planned on the host: the copy is made once per
    tensor and refreshed only when the tensor changes in place, so callers
    that keep their tables (as the reference's models keep buffers) pay no
    device-to-host copy per call."""
    from kernel import fused_attn as F
    t = torch.tensor([0, 2, 1, 0], dtype=torch.int32)
    a = F._host_table(t)
    assert a.tolist() == [0, 2, 1, 0]
    assert F._host_table(t) is a                      # cached on the tensor
    t[1] = 1                                          # in-place change: version moves
    b = F._host_table(t)
    assert b.tolist() == [0, 1, 1, 0]
    assert F._host_table(t.clone()) is not b          # another tensor: its own copy
    assert F._host_table(None) is None
    assert F._host_table([1, 2]).tolist() == [1, 2]


def test_close_rows_refused():
    """16-bit rows closer than the head dim, which the kernels' descriptors cut
    short, are refused where they would be read so; one row has no pitch."""
    L = _ext.lib()
    for name in ("k", "v"):
        a = _args()
        getattr(a, name).stride[2] = 0
        assert L.saf_mixed_attn_fwd(ctypes.byref(a), None) == _ext.SAF_EALIGN
        assert "closer than" in L.saf_last_error().decode()
    d, p = (_ext.SafTensor.from_buffer_copy(_args().v) for _ in range(2))
    d.stride[2] = 32
    p.ndim, p.dtype = 3, _ext.SAF_F32
    for i, n in enumerate((4, 64, 64)):
        p.size[i], p.stride[i] = n, (4096, 64, 1)[i]
    fz = (ctypes.c_int32 * 4)(0, 1, 2, 3)
    out = _args().v
    assert L.saf_frozen_pv_bwd(p, d, fz, 4, 64, out, None) == _ext.SAF_EALIGN
    assert L.saf_frozen_pv_fwd(p, d, fz, 4, 64, out, None) == _ext.SAF_EALIGN


def test_cpu_table_sharing_memory():
    """A routing table on the CPU that shares memory with numpy: an edit through
    numpy moves no version, and both the host copy and its ctypes twin follow."""
    import numpy as np
    from kernel import fused_attn as F
    arr = np.array([0, 2, 1, 0], dtype=np.int32)
    t = torch.from_numpy(arr)
    for states in ([0, 2, 1, 0], [2, 0, 0, 1]):
        arr[:] = states
        host, twin = F._table(t)
        assert host.tolist() == states and list(twin) == states


@pytest.mark.parametrize("hd,B,T,n_live,n_dec,n_scan,asked,want", [
    (64, 1, 1024, 1, 2, 0, 0, 0),
    (64, 1, 1024, 1, 2, 1, 1, 3),      # asked for: the scan goes along
    (64, 8, 4096, 9, 3, 0, 0, 1),      # hd 64: the live heads outlast a decomposed walk
    (64, 8, 4096, 9, 3, 0, -1, 0),
    (64, 4, 4096, 9, 3, 0, 0, 0),
    (64, 8, 2048, 9, 3, 0, 0, 0),
    (64, 8, 3001, 9, 3, 1, 0, 3),
    (32, 8, 3000, 9, 3, 0, 0, 1),
    (128, 4, 2048, 9, 3, 0, 0, 1),     # hd 128: CUs are left without a live workgroup
    (128, 1, 1024, 9, 3, 0, 0, 0),
    (128, 8, 4096, 9, 3, 0, 0, 0),
    (96, 2, 4096, 9, 3, 0, 0, 1),
    (256, 1, 1024, 9, 3, 0, 0, 1),
    (256, 2, 4096, 9, 3, 0, 0, 0),
    (64, 8, 4096, 1, 0, 1, 0, 0),      # 40 us of live heads
    (64, 8, 16384, 1, 0, 1, 0, 2),
    (64, 8, 16384, 1, 1, 1, -1, 2),
])
def test_side_kernels(hd, B, T, n_live, n_dec, n_scan, asked, want):
    """Which kernels leave the caller's stream: one rule for the call and for
    the per-kind schedule that is timed."""
    H = n_live + n_dec + n_scan
    a = _args(H=H, T=T, hd=hd, frozen=[0] * n_live + [2] * (n_dec + n_scan))
    for t in (a.q, a.k, a.v, a.out):
        t.size[0] = B
    for t in (a.alpha, a.rho, a.z):
        t.data, t.dtype, t.ndim = 0x100000, _ext.SAF_F32, 2
        t.size[0], t.size[1], t.stride[0], t.stride[1] = H, T, T, 1
    kinds = (ctypes.c_int32 * H)(*[0] * (n_live + n_dec), *[1] * n_scan)
    prm = (ctypes.c_float * H)()
    a.closed_kind, a.closed_param, a.decomp_unsplit = kinds, prm, asked
    assert _ext.lib().saf_mixed_attn_side_kernels(ctypes.byref(a)) == want
    a.n_heads = 0
    assert _ext.lib().saf_mixed_attn_side_kernels(ctypes.byref(a)) == -1


def _split_bytes(state, H, T, hd, B=1, patt_dtype=_ext.SAF_F32, pitch=None):
    """Workspace of H heads of one state beyond what every length of it needs:
    the partials of split query blocks (a plan that does not split has none)."""
    a = _args(H=H, T=T, hd=hd, frozen=[state] * H)
    for t in (a.q, a.k, a.v, a.out):
        t.size[0] = B
    for t in (a.alpha, a.rho, a.z):
        t.data, t.dtype, t.ndim = 0x100000, _ext.SAF_F32, 2
        t.size[0], t.size[1], t.stride[0], t.stride[1] = H, T, T, 1
    pitch = pitch or T
    a.patt.data, a.patt.dtype, a.patt.ndim = 0x100000, patt_dtype, 3
    for i, (n, st) in enumerate(((H, pitch * T), (T, pitch), (T, 1))):
        a.patt.size[i], a.patt.stride[i] = n, st
    n = _ext.lib().saf_mixed_attn_workspace_bytes(ctypes.byref(a))
    assert n >= 0
    return n


@pytest.mark.parametrize("B,H,T", [(1, 12, 2048), (4, 3, 2048), (1, 12, 4096), (1, 3, 8192)])
def test_decomposed_hd256_splits(B, H, T):
    """Decomposed heads of hd 256 rebuild P cell by cell: their long query blocks
    are split where those of hd 128 may not be (half the time at these shapes)."""
    assert _split_bytes(2, H, T, 256, B) > 0


@pytest.mark.parametrize("B,H,T,hd", [(8, 3, 3001, 64), (4, 8, 4097, 128), (1, 3, 2049, 256)])
@pytest.mark.parametrize("dtype", [_ext.SAF_BF16, _ext.SAF_F16, _ext.SAF_F32])
def test_dense_patterns_of_odd_pitch_split(B, H, T, hd, dtype):
    """Patterns that are read element by element (rows off 16-byte boundaries)
    cost several times the fast forms' block: their long query blocks are split."""
    assert _split_bytes(1, H, T, hd, B, patt_dtype=dtype, pitch=T) > 0


def test_aligned_view_keeps_what_both_rules_accept():
    """_aligned_view's one pass over shape and strides against the two rules it
    stands for, over strides, sizes of one, offsets and types."""
    import random
    from kernel import fused_attn as F
    r = random.Random(1)
    for _ in range(3000):
        shape = [r.choice([1, 2, 3]) for _ in range(3)] + [r.choice([1, 32, 64])]
        stride = [r.choice([0, 1, 8, 16, 24, 32, 64, 65, 72, 128, 4096]) for _ in range(3)] + [r.choice([0, 1, 2])]
        base = torch.zeros(30000, dtype=r.choice([torch.bfloat16, torch.float32]))
        x = base.as_strided(shape, stride, r.choice([0, 1, 8]))
        kept = F._aligned_view(x, 16) is x
        # contiguous() returns a tensor that counts as contiguous already
        assert kept == (F._row_aligned(x, 16) and F._rows_apart(x)) or x.is_contiguous(), (shape, stride)
