"""Build libhilberta_hip.so (gfx950, hipcc) and libhilberta_torch.so (the torch operators) in-tree.

    python -m hilberta_amd.build          # compile every csrc/*.hip and torch_ops.cpp, link both

Objects go to hilberta_amd/_build/, the libraries to hilberta_amd/; all are git-ignored.
libhilberta_torch.so is host code over the C ABI, built against the installed torch.
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OUT = PKG / "_build"
LIB = PKG / "libhilberta_hip.so"
TORCH_LIB = PKG / "libhilberta_torch.so"
TORCH_SRC = CSRC / "torch_ops.cpp"
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-variable",
    "-Wno-unused-lambda-capture",
    # packed fp32 VALU ops stay off: the compiler must not emit v_pk_{add,mul,fma}_f32
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-munsafe-fp-atomics",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found: the HIP toolchain (ROCm) is required to build")


# Per-file flags.  attention.hip: no atomic optimizer.  Its atomics are single-lane work-queue
# claims; the optimizer turns each into a wave-aggregated atomic that reads its result back (and
# so waits for the round trip) right after issue, where the kernel means to overlap it with a step.
FILE_FLAGS = {"attention.hip": ["-mllvm", "-amdgpu-atomic-optimizer-strategy=None"]}


def _compile(src: Path) -> Path:
    obj = OUT / (src.stem + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, *FILE_FLAGS.get(src.name, []), "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(line for line in proc.stderr.splitlines() if noise not in line)
    if proc.returncode:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{err}")
    if err.strip():
        print(err, file=sys.stderr)
    return obj


def _host_compiler() -> str:
    for cand in (os.environ.get("CXX"), shutil.which("g++"), shutil.which("c++")):
        if cand and shutil.which(cand):
            return cand
    raise RuntimeError("a host C++ compiler (g++) is required to build the torch operators")


def _run(cmd, what):
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode:
        raise RuntimeError(f"{what} failed:\n{proc.stderr}")


def _compile_torch_ops() -> Path:
    import torch
    from torch.utils.cpp_extension import include_paths

    obj = OUT / (TORCH_SRC.stem + ".o")
    includes = [arg for path in include_paths("cuda") for arg in ("-isystem", path)]
    _run([_host_compiler(), "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *includes, "-c", str(TORCH_SRC),
          "-o", str(obj)], f"compiling {TORCH_SRC.name}")
    return obj


def _link_torch_ops(obj: Path) -> None:
    """Against the library beside it ($ORIGIN) and the installed torch, which is loaded before it."""
    from torch.utils.cpp_extension import library_paths

    tmp = TORCH_LIB.with_suffix(".so.tmp")
    _run([_host_compiler(), "-shared", str(obj), "-o", str(tmp), f"-L{PKG}", f"-l:{LIB.name}", "-Wl,-rpath,$ORIGIN",
          *(f"-L{path}" for path in library_paths("cuda")), "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip"],
         f"linking {TORCH_LIB.name}")
    os.replace(tmp, TORCH_LIB)


def build(verbose: bool = True) -> Path:
    OUT.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(sources))) as pool:
        torch_ops = pool.submit(_compile_torch_ops)
        objects = list(pool.map(_compile, sources))
        torch_object = torch_ops.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objects), "-o", str(tmp)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode:
        raise RuntimeError(f"link failed:\n{proc.stderr}")
    # a kernel whose host-side launch stub was not emitted links fine but cannot be loaded
    undefined = subprocess.run(["nm", "-D", "--undefined-only", str(tmp)], capture_output=True,
                               text=True).stdout
    stubs = [line.split()[-1] for line in undefined.splitlines() if "__device_stub__" in line]
    if stubs:
        raise RuntimeError(f"link left {len(stubs)} kernel launch stubs undefined, e.g. {stubs[0]}")
    os.replace(tmp, LIB)
    _link_torch_ops(torch_object)
    if verbose:
        print(f"built {LIB} from {len(sources)} sources, and {TORCH_LIB.name}")
    return LIB


if __name__ == "__main__":
    build()
