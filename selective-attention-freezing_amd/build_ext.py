"""Builds libsafattn.so in-tree for gfx950 with hipcc.

Objects go to ``_build/`` beside this file, the shared library to
``kernel/libsafattn.so``.  Every call recompiles (the build check of the
driver must exercise the compiler).
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
OUT = os.path.join(HERE, "kernel", "libsafattn.so")
SOURCES = ("saf_capi.hip", "flash_fwd.hip", "frozen_pv.hip", "frozen_scan.hip", "rope.hip", "layernorm.hip",
           "attn_bwd.hip", "decomp_logz.hip", "attn_f32.hip", "proj_gemm.hip")
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # packed-fp32 instructions are kept out of every kernel (the compiler
    # still emits scalar fp32 FMA/MUL); hipcc's host pass ignores the feature
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(REPO, "include"), "-I", CSRC,
]


# Per-source flags.  The backward kernels keep four MFMA accumulator sets
# alive across their loops; with the default AGPR form the compiler parks
# them in VGPRs and copies every one into AGPRs and back around each product
# (hundreds of v_accvgpr moves per query block).  The VGPR form of the MFMA
# instructions removes the copies and lowers register use.  The float32
# kernels hold their accumulators across loops the same way.
SOURCE_FLAGS = {"attn_bwd.hip": ("-mllvm", "-amdgpu-mfma-vgpr-form"),
                "attn_f32.hip": ("-mllvm", "-amdgpu-mfma-vgpr-form")}


def _hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.sep not in cand or os.path.exists(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _run(cmd):
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    lines = [ln for ln in res.stdout.splitlines()
             if "packed-fp32-ops" not in ln and "is not a recognized feature" not in ln]
    if res.returncode != 0:
        raise RuntimeError("build failed: " + " ".join(cmd) + "\n" + "\n".join(lines))
    return "\n".join(lines)


def build(verbose=False, jobs=None):
    """Compile every HIP source for gfx950 and link kernel/libsafattn.so."""
    os.makedirs(BUILD, exist_ok=True)
    hipcc = _hipcc()
    objs = []
    cmds = []
    for src in SOURCES:
        obj = os.path.join(BUILD, src.replace(".hip", ".o"))
        objs.append(obj)
        cmds.append([hipcc, *HIPCC_FLAGS, *SOURCE_FLAGS.get(src, ()), "-c", os.path.join(CSRC, src), "-o", obj])
    jobs = jobs or min(len(cmds), max(1, os.cpu_count() or 1))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        for out in ex.map(_run, cmds):
            if verbose and out:
                print(out)
    tmp = OUT + ".tmp"
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs])
    os.replace(tmp, OUT)
    if verbose:
        print(f"built {OUT}")
    return OUT


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
