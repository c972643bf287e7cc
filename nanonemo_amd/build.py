"""Ahead-of-time build of the HIP library for gfx950.

Replaces the reference's JIT build (/root/reference/nanonemo/kernels/cuda/__init__.py:15-18, which runs
nvcc through torch.utils.cpp_extension.load on first use): here ``hipcc`` compiles
``nanonemo_amd/csrc/*.hip`` once, in-tree, into ``nanonemo_amd/lib/libnanonemo_fa.so``, a plain C-ABI
shared library with no torch types in its signatures (include/*.h), and ``g++`` compiles ``csrc/host.cpp`` into
``nanonemo_host.so``, the torch extension that calls it.

    python -m nanonemo_amd.build
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
SRCS = [PKG / "csrc" / f"{n}.hip" for n in ("flash_attn", "rope", "rmsnorm", "linear", "loss")]
LIB_DIR = PKG / "lib"
LIB = LIB_DIR / "libnanonemo_fa.so"
# Block timelines for `bench.py --timeline`: the attention kernels built with NN_TIMELINE=1, so that every block
# records clock stamps at its phase boundaries (the product library compiles those stamps to nothing).
TIMELINE_SRCS = [PKG / "csrc" / "flash_attn.hip"]
TIMELINE_LIB = LIB_DIR / "libnanonemo_fa_timeline.so"
ARCH = "gfx950"

# -packed-fp32-ops: keep v_pk_{add,mul,fma}_f32 out of the generated code (those packed forms have
# produced intermittent wrong results on the target boxes). hipcc's host pass warns that it does not
# know the feature; that warning is harmless.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    # Select MFMAs in their VGPR form and let register allocation move accumulators to AGPRs where it
    # must: the dK / dV kernel then keeps dK^T / dV^T in AGPRs while S and dP stay in VGPRs, where
    # the softmax reads them, instead of copying every S / dP element out of an AGPR (2-3 % faster;
    # no other kernel's code changes).
    "-mllvm",
    "-amdgpu-mfma-vgpr-form=1",
    # The first 16 dwords of a kernel's arguments arrive in scalar registers with the launch instead of by a scalar load
    # at its start: the forward 1.5-3 % faster at B=1-32, T=256-512, other kernels and shapes within noise.
    "-mllvm",
    "-amdgpu-kernarg-preload-count=16",
]
# Device code never relies on NaN semantics (masked scores are -inf, never NaN), except the cross entropy's, which
# must show NaN and infinite logits; without this every fmaxf of an MFMA result is preceded by a canonicalising
# v_max_f32 x, x.
NO_NANS = ["-Xarch_device", "-fno-honor-nans"]
HONOR_NANS = {"loss"}


# The host side of the operations, a torch extension over the library (g++: it has no device code).
HOST_SRC = PKG / "csrc" / "host.cpp"
HOST_LIB = LIB_DIR / "nanonemo_host.so"


def _host_command(out: str) -> list[str]:
    """Compile the host module; it links the library beside it."""
    import sysconfig

    import torch

    base = Path(torch.__file__).resolve().parent
    rocm = Path(hipcc()).resolve().parents[1]
    includes = [base / "include", base / "include" / "torch" / "csrc" / "api" / "include", rocm / "include", sysconfig.get_paths()["include"]]
    libs = ["c10", "c10_hip", "torch", "torch_cpu", "torch_hip", "torch_python"]
    return [
        "g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
        "-DTORCH_EXTENSION_NAME=nanonemo_host", "-DTORCH_API_INCLUDE_EXTENSION_H", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
        *(a for p in includes for a in ("-isystem", str(p))), f"-I{ROOT / 'include'}", "-o", out, str(HOST_SRC),
        f"-L{base / 'lib'}", f"-L{LIB_DIR}", "-lnanonemo_fa", *(f"-l{n}" for n in libs), "-Wl,-rpath,$ORIGIN",
    ]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (looked at $HIPCC, /opt/rocm/bin/hipcc and PATH)")


def _run(cmd: list[str], verbose: bool) -> None:
    """One compiler command; raises with its output if it fails."""
    if verbose:
        print(" ".join(cmd), flush=True)
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    noise = "'-packed-fp32-ops' is not a recognized feature"
    log = "\n".join(l for l in p.stdout.splitlines() if noise not in l)
    if p.returncode != 0:
        raise RuntimeError(f"{Path(cmd[0]).name} failed ({p.returncode}): {' '.join(cmd)}\n{log}")
    if verbose and log.strip():
        print(log, flush=True)


def build(verbose: bool = False) -> Path:
    """Compile the HIP library, the timeline build of the attention kernels and the host module, the HIP sources in
    parallel (always recompiles); return the library's path."""
    LIB_DIR.mkdir(parents=True, exist_ok=True)
    with tempfile.TemporaryDirectory() as tmp, ThreadPoolExecutor() as pool:
        jobs = []
        for lib, srcs, defines in ((LIB, SRCS, []), (TIMELINE_LIB, TIMELINE_SRCS, ["-DNN_TIMELINE=1"])):
            for src in srcs:
                obj = str(Path(tmp) / f"{lib.stem}_{src.stem}.o")
                flags = [*HIPCC_FLAGS, *([] if src.stem in HONOR_NANS else NO_NANS), *defines]
                cmd = [hipcc(), "-c", *flags, f"-I{ROOT / 'include'}", "-o", obj, str(src)]
                jobs.append((lib, obj, pool.submit(_run, cmd, verbose)))
        errors = [str(e) for e in (job.exception() for _, _, job in jobs) if e]
        if errors:
            raise RuntimeError("\n".join(errors))
        for lib in (LIB, TIMELINE_LIB):
            out = lib.with_suffix(".so.tmp")
            _run([hipcc(), f"--offload-arch={ARCH}", "-shared", "-o", str(out), *(obj for to, obj, _ in jobs if to == lib)], verbose)
            os.replace(out, lib)  # atomic: a process that already mapped the old file keeps it
    out = HOST_LIB.with_suffix(".so.tmp")
    _run(_host_command(str(out)), verbose)
    os.replace(out, HOST_LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-q" not in sys.argv))
