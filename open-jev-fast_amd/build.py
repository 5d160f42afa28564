"""Builds libojx.so (the HIP kernels + C-ABI of the projection path) in-tree for gfx950 with hipcc.

Run as `python open-jev-fast_amd/build.py` or through `__graft_entry__.build()`. The library lands next to this file
so that it travels with the source tree; nothing is installed.
"""
import hashlib
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")
LIB = os.path.join(HERE, "libojx.so")
SOURCES = ["gemm.hip", "gemm_sk.hip", "gemm_kx_a.hip", "gemm_kx_b.hip", "gemm_kx_c.hip", "epilogue.hip", "prep.hip", "api.hip"]
OBJDIR = os.path.join(HERE, "_build")
ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# -packed-fp32-ops off: hipcc would otherwise fuse float pairs into v_pk_{add,mul,fma}_f32, which this fleet
# must not run. The host pass warns that it does not know the feature; that warning is expected.
FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         # the fragment epilogues must unroll completely, or the accumulator array is left in scratch memory
         "-mllvm", "-pragma-unroll-threshold=1000000",
         f"-I{INCLUDE}", f"-I{CSRC}"]


def source_files():
    """Every file the library is compiled from: csrc/ (kernels, C-ABI, plan table) and include/ojx.h."""
    files = [os.path.join(CSRC, f) for f in sorted(os.listdir(CSRC))
             if f.endswith((".hip", ".h", ".inc"))]
    return files + [os.path.join(INCLUDE, "ojx.h")]


def source_digest() -> str:
    """sha256 (first 16 hex digits) over the names and bytes of source_files(). It is compiled into the library
    (ojx_version() ends in "src:<digest>"), so a loaded libojx.so can be checked against the tree beside it."""
    h = hashlib.sha256()
    for f in source_files():
        h.update(os.path.basename(f).encode() + b"\0")
        with open(f, "rb") as fh:
            h.update(fh.read())
        h.update(b"\0")
    return h.hexdigest()[:16]


def build(verbose: bool = False) -> str:
    """Compiles every source into libojx.so (always rebuilds; the translation units compile in parallel).
    Returns the library path."""
    os.makedirs(OBJDIR, exist_ok=True)
    noise = "is not a recognized feature for this target"
    jobs = []
    digest = source_digest()
    for s in SOURCES:
        obj = os.path.join(OBJDIR, s.replace(".hip", ".o"))
        cmd = [HIPCC, *FLAGS, f'-DOJX_SRC_DIGEST="{digest}"', "-c", os.path.join(CSRC, s), "-o", obj]
        jobs.append((cmd, obj, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)))
    errs = []
    for cmd, obj, pr in jobs:
        _, err = pr.communicate()
        err = "\n".join(l for l in err.splitlines() if noise not in l)
        if pr.returncode != 0:
            errs.append(f"hipcc failed ({pr.returncode}):\n{' '.join(cmd)}\n{err}")
        elif verbose and err.strip():
            print(err, file=sys.stderr)
    if errs:
        raise RuntimeError("\n".join(errs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", f"--offload-arch={ARCH}", *[o for _, o, _ in jobs], "-o", tmp]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed ({res.returncode}):\n{' '.join(cmd)}\n{res.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
