"""Build recipe for ``libnf_cdna4.so`` (the C-ABI library of hand-written gfx950 kernels).

``python -m triton_helpers_amd.build`` cross-compiles every ``csrc/*.hip`` with
``hipcc --offload-arch=gfx950`` (no GPU needed) and links them into
``triton_helpers_amd/libnf_cdna4.so`` next to this file, then compiles the host side of the
operators (``csrc/host_native.cpp``) into ``triton_helpers_amd/_native.so``.
"""
from __future__ import annotations

import os
import re
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path
from typing import List, Sequence

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
INCLUDE = PKG_DIR.parent / "include"
LIB_PATH = PKG_DIR / "libnf_cdna4.so"
BUILD_DIR = PKG_DIR / "build"
NATIVE_PATH = PKG_DIR / "_native.so"

ARCH = "gfx950"
# Features of the GPU target that are switched off.  hipcc hands them to its host pass as well, which says that it does not know them.
NO_PACKED_FP32, NO_MERGED_LDS = "-packed-fp32-ops", "-load-store-opt"


def _feature(name: str) -> List[str]:
    return ["-Xclang", "-target-feature", "-Xclang", name]


def _unknown(name: str) -> str:
    return f"'{name}' is not a recognized feature for this target (ignoring feature)"


COMMON_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-munsafe-fp-atomics",
    # keep the compiler from emitting packed-fp32 VALU forms
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{INCLUDE}",
    f"-I{CSRC}",
]
# Files whose float arithmetic must not be contracted into FMAs (bit-exact cell / weight math).
NO_CONTRACT = {"hash_encoding.hip", "hash_encoding_bwd_scan.hip", "hash_encoding_bwd_bin.hip", "hash_encoding_bwd_static.hip", "hash_check_host.hip"}
# Files whose MFMA results feed vector ALU work directly: keep them in architectural VGPRs instead of
# bouncing every result through an accumulation register.
MFMA_VGPR_FORM = {"fused_mlp.hip", "fused_mlp_bwd2.hip", "fused_mlp_bwdn.hip", "fused_mlp_bwd2_w8.hip", "fused_mlp_bwd2_ws.hip", "fused_mlp_bwd_roles.hip", "fused_mlp_fwd2.hip", "reversible_mlp.hip", "reversible_bwd.hip"}
# Files whose LDS reads stay as written: merged in pairs (ds_read2st64_b64) they take 2.6 times as long on this chip (12 against 4.5 clocks of
# the kernel's timer, two reads of 512 bytes), and almost five times where the single ones are free of bank conflicts.
SINGLE_READS = {"fused_mlp_bwd_roles.hip", "reversible_bwd.hip"}
# Kernels at the edge of the register file (their gradient waves hold up to 128 sums of 168 registers, or 160 of 256) that must not spill: a
# spilled sum is read and written in every section, and the compiler has got one wrong in a kernel of this kind (it set the high half of a
# 64-bit row counter aside in an accumulation register and never read it back).
NO_SPILL = {"reversible_bwd.hip": "rev_bwd_k", "fused_mlp_bwd_roles.hip": "mlp_bwd_roles_k"}


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; a ROCm toolchain is required to build libnf_cdna4.so")
    return exe


def _run(cmd: List[str], verbose: bool) -> str:
    if verbose:
        print("+", " ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if l not in (_unknown(NO_PACKED_FP32), _unknown(NO_MERGED_LDS)))
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
    if verbose and out.strip():
        print(out, flush=True)
    return out


def check_features(hipcc: str, names: Sequence[str] = (NO_PACKED_FP32, NO_MERGED_LDS)) -> None:
    """Refuse a compiler whose GPU pass does not know one of the features: it would only say so, and ignore the flag."""
    flags = [f for name in names for f in _feature(name)]
    cmd = [hipcc, f"--offload-arch={ARCH}", "--offload-device-only", *flags, "-x", "hip", "-c", os.devnull, "-o", os.devnull]
    out = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True).stdout
    unknown = [name for name in names if _unknown(name) in out]
    if unknown:
        raise RuntimeError(f"{hipcc} does not know {', '.join(unknown)} for {ARCH}")


def _check_spills(out: str, kernel: str) -> None:
    """Refuse a build whose resource remarks show spilled registers in ``kernel``."""
    seen = 0
    for part in out.split("Function Name: ")[1:]:
        name, spill = part.split()[0], re.search(r"VGPRs Spill: (\d+)", part)
        if kernel in name:
            seen += 1
            if spill is None or int(spill[1]) != 0:
                raise RuntimeError(f"{name} spills registers; its listing has to be looked through before it may run")
    if not seen:
        raise RuntimeError(f"no resource remarks for {kernel}")


def _compile(cmd: List[str], src: Path, verbose: bool) -> None:
    kernel = NO_SPILL.get(src.name)
    if kernel is None:
        _run(cmd, verbose)
    else:
        _check_spills(_run([*cmd, "-Rpass-analysis=kernel-resource-usage"], False), kernel)


def sources() -> List[Path]:
    return sorted(CSRC.glob("*.hip"))


def native_command(out: Path) -> List[str]:
    """The operators' host side: a CPython module on torch's headers, linked to the kernel library beside it."""
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        raise RuntimeError("a C++ compiler is required to build _native.so")
    rocm = Path(_hipcc()).resolve().parent.parent
    includes = [*include_paths(), str(rocm / "include"), sysconfig.get_paths()["include"]]
    return [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{INCLUDE}", *(f"-isystem{d}" for d in includes),
            str(CSRC / "host_native.cpp"), "-o", str(out), f"-L{PKG_DIR}", f"-l:{LIB_PATH.name}", *(f"-L{d}" for d in library_paths()),
            "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]


def build(verbose: bool = True, jobs: int = 8) -> Path:
    """Compile all kernels, link the shared library and the native host module on it; returns the library's path."""
    hipcc = _hipcc()
    check_features(hipcc)
    BUILD_DIR.mkdir(exist_ok=True)
    objs = []
    cmds = []
    for src in sources():
        obj = BUILD_DIR / (src.stem + ".o")
        flags = list(COMMON_FLAGS)
        if src.name in NO_CONTRACT:
            flags.append("-ffp-contract=off")
        if src.name in MFMA_VGPR_FORM:
            flags += ["-mllvm", "-amdgpu-mfma-vgpr-form"]
        if src.name in SINGLE_READS:
            flags += _feature(NO_MERGED_LDS)
        cmds.append(([hipcc, *flags, "-c", str(src), "-o", str(obj)], src))
        objs.append(obj)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        list(ex.map(lambda c: _compile(*c, verbose), cmds))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)], verbose)
    os.replace(tmp, LIB_PATH)
    tmp = NATIVE_PATH.with_suffix(".so.tmp")
    _run(native_command(tmp), verbose)
    os.replace(tmp, NATIVE_PATH)
    return LIB_PATH


if __name__ == "__main__":
    path = build(verbose="-q" not in sys.argv)
    print(f"built {path}")
