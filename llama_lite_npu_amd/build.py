"""Builds liblitekv.so (HIP, gfx950) in-tree with hipcc, and the Python module of the calls that take
PyTorch tensors (host code) with g++.

Usage: ``python -m llama_lite_npu_amd.build`` or ``build_library(force=True)``.
hipcc cross-compiles for gfx950 without a GPU, so this also runs on a CPU-only
machine. The library lands next to its sources (``csrc/liblitekv.so``), the module in the
package; nothing is installed outside the tree.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

CSRC = Path(__file__).resolve().parent / "csrc"
LIB_PATH = CSRC / "liblitekv.so"
# csrc/torch_calls.cpp; the suffix names the interpreter it is for, and another one does not find it
CALLS_PATH = CSRC.parent / f"_calls{sysconfig.get_config_var('EXT_SUFFIX') or '.so'}"
OBJ_DIR = CSRC / "build"

SOURCES = (
    "status.hip",
    "kv_append.hip",
    "kv_fp8.hip",
    "qk_rope_append.hip",
    "page_ops.hip",
    "paged_decode.hip",
    "paged_decode_hd64.hip",
    "decode_advance.hip",
    "copy_segments.hip",
    "paged_prefill.hip",
    "paged_prefill_hd64.hip",
    "paged_prefill_hd256.hip",
    "generic_attention.hip",
)

# Packed fp32 VALU forms are switched off for device code: the compiler would
# otherwise form them on its own from scalar float arithmetic.
HIPCC_FLAGS = (
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
)


# Extra flags per source. The prefill kernel takes maxima of MFMA results: without NaN
# semantics to honour, the compiler drops the self-max that quiets each operand and fuses the
# rest into v_max3_f32. Nothing in that file relies on NaN propagation (masking uses -inf).
# Its direct HBM -> LDS loads set m0 in inline assembly and list it as clobbered; the compiler
# remarks on every such statement that m0 is a reserved register, which is the point of listing it.
PER_FILE_FLAGS = {
    "paged_prefill.hip": ("-fno-honor-nans", "-Wno-inline-asm"),
    "paged_prefill_hd64.hip": ("-fno-honor-nans", "-Wno-inline-asm"),
    # at head dim 256 not a number goes where fp32 arithmetic takes it: no NaN flag (231 more
    # v_max_f32 in its four kernels, none in the loop over tiles below the diagonal)
    "paged_prefill_hd256.hip": ("-Wno-inline-asm",),
    # the decode step behind a shared prefix runs the same tile kernel as one role of its launch
    "paged_decode.hip": ("-Wno-inline-asm",),
    "paged_decode_hd64.hip": ("-Wno-inline-asm",),
}


def _hipcc() -> str:
    found = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(found):
        raise RuntimeError("hipcc not found; liblitekv needs the ROCm toolchain to build")
    return found


def _headers() -> list[Path]:
    return sorted(CSRC.glob("*.h")) + sorted(CSRC.glob("*.inc")) + sorted((CSRC.parents[1] / "include").glob("*.h"))


def is_stale() -> bool:
    if not LIB_PATH.exists():
        return True
    built = LIB_PATH.stat().st_mtime
    deps = [CSRC / s for s in SOURCES] + _headers()
    return any(d.stat().st_mtime > built for d in deps)


def _compile(hipcc: str, src: Path, obj: Path, extra: tuple[str, ...]) -> None:
    cmd = [hipcc, *HIPCC_FLAGS, *extra, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "'-packed-fp32-ops' is not a recognized feature"
    log = "\n".join(l for l in (proc.stdout + proc.stderr).splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{log}")
    if log.strip():
        print(log, file=sys.stderr)


def build_library(force: bool = False, extra_flags: tuple[str, ...] = ()) -> Path:
    """Compiles every source and links liblitekv.so, then the module of the tensor calls; returns the
    library's path."""
    if not force and not is_stale():
        build_calls()
        return LIB_PATH
    hipcc = _hipcc()
    OBJ_DIR.mkdir(exist_ok=True)
    objs = [OBJ_DIR / (Path(s).stem + ".o") for s in SOURCES]
    with ThreadPoolExecutor(max_workers=min(len(SOURCES), 8)) as pool:
        jobs = [
            pool.submit(_compile, hipcc, CSRC / s, o, PER_FILE_FLAGS.get(s, ()) + tuple(extra_flags))
            for s, o in zip(SOURCES, objs)
        ]
        for j in jobs:
            j.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link of liblitekv.so failed:\n{proc.stdout}{proc.stderr}")
    os.replace(tmp, LIB_PATH)
    build_calls(force)
    return LIB_PATH


def build_calls(force: bool = False) -> Path:
    """Compiles the Python module of the calls that take PyTorch tensors (host code, no kernel); returns its
    path. It finds liblitekv.so next to its source."""
    src = CSRC / "torch_calls.cpp"
    deps = [src, CSRC.parents[1] / "include" / "litekv.h"]
    if not force and CALLS_PATH.exists() and all(d.stat().st_mtime <= CALLS_PATH.stat().st_mtime for d in deps):
        return CALLS_PATH
    import torch
    from torch.utils import cpp_extension

    torch_lib = Path(torch.__file__).resolve().parent / "lib"
    includes = [CSRC.parents[1] / "include", sysconfig.get_paths()["include"], *cpp_extension.include_paths()]
    tmp = CALLS_PATH.with_name(CALLS_PATH.name + ".tmp")
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-isystem{i}" for i in includes),
           str(src), "-o", str(tmp), f"-L{torch_lib}", "-ltorch_python", "-ltorch_cpu", "-lc10",
           f"-L{CSRC}", f"-l:{LIB_PATH.name}", f"-Wl,-rpath,$ORIGIN/{CSRC.name}"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"build of {CALLS_PATH.name} failed:\n{proc.stdout}{proc.stderr}")
    os.replace(tmp, CALLS_PATH)
    return CALLS_PATH


if __name__ == "__main__":
    print(build_library(force=True))
    print(CALLS_PATH)
