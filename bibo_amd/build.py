"""Build recipe: every .hip file under csrc/ compiled for gfx950 with hipcc and linked into libbibo_moe.so next to this file,
and csrc/binding.cpp compiled with g++ into _native.so, the modules' host path over that library.
`python -m bibo_amd.build` runs it."""
from __future__ import annotations

import os
import pathlib
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = pathlib.Path(__file__).resolve().parent
CSRC = HERE / "csrc"
BUILD = HERE / "csrc" / "build"
LIB = HERE / "libbibo_moe.so"
NATIVE = HERE / "_native.so"

# longest first
SOURCES = ["experts_fused_384.hip", "experts_fused_256.hip", "experts_fused_128.hip", "experts_fused_512.hip", "backward.hip", "router.hip", "backward_generic.hip",
           "experts_generic.hip", "experts_mfma.hip", "exp_attention.hip", "experts_stream.hip", "experts_few.hip", "ffn.hip", "permute.hip",
           "experts_fused.hip", "api.hip"]

# -packed-fp32-ops is switched off on purpose: hipcc -O3 otherwise forms v_pk_*_f32 from scalar float code.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-warning-option",
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: the HIP extension cannot be built on this machine")
    return exe


def _compile(src: str, extra: list[str]) -> pathlib.Path:
    obj = BUILD / (src + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, *extra, "-c", str(CSRC / src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    if r.stderr.strip():
        # the host pass warns that it does not know -packed-fp32-ops; that is harmless
        lines = [l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip()]
        if lines:
            sys.stderr.write("\n".join(lines) + "\n")
    return obj


def _run(cmd: list[str], what: str) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{r.stdout}\n{r.stderr}")


def _compile_binding() -> pathlib.Path:
    import torch
    from torch.utils import cpp_extension
    obj = BUILD / "binding.cpp.o"
    includes = [f"-I{p}" for p in (*cpp_extension.include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include")]
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM", "-DTORCH_EXTENSION_NAME=_native",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *includes, "-c", str(CSRC / "binding.cpp"), "-o",
          str(obj)], "g++ on binding.cpp")
    return obj


def _link_binding(obj: pathlib.Path) -> None:
    import torch
    lib_dir = pathlib.Path(torch.__file__).parent / "lib"
    tmp = NATIVE.with_suffix(".so.tmp")
    _run(["g++", "-shared", "-fPIC", str(obj), "-o", str(tmp), f"-L{lib_dir}", "-ltorch", "-ltorch_python", "-ltorch_cpu", "-lc10",
          "-lc10_hip", f"-L{HERE}", "-lbibo_moe", "-Wl,-rpath,$ORIGIN"], "link of _native.so")
    os.replace(tmp, NATIVE)


def build(extra_flags: list[str] | None = None, jobs: int = 6) -> pathlib.Path:
    """Compile every source and link the shared library and the native binding; always recompiles."""
    BUILD.mkdir(parents=True, exist_ok=True)
    extra = list(extra_flags or [])
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        binding = ex.submit(_compile_binding)
        objs = list(ex.map(lambda s: _compile(s, extra), SOURCES))
        binding_obj = binding.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    _run(cmd, "link")
    os.replace(tmp, LIB)
    _link_binding(binding_obj)
    return LIB


if __name__ == "__main__":
    print(build(sys.argv[1:]))
