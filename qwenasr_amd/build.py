"""Build recipe for the gfx950 kernel library.

Compiles every ``csrc/*.hip`` with hipcc for gfx950 and produces, in-tree:

* ``qwenasr_amd/libqasr_hip.so`` -- shared library the Python and C++ hosts load;
* ``qwenasr_amd/_binding.so``     -- the Python extension through which ``kernels.py``
  calls it (host code only, against torch's and Python's headers; without these the
  libraries are built alone, and a line says so);
* ``qwenasr_amd/libqasr_hip.a``  -- static archive for a host that links it
  statically (a Rust ``build.rs`` would add ``cargo:rustc-link-lib=static=qasr_hip``
  plus ``amdhip64``).

Run ``python -m qwenasr_amd.build`` (or ``__graft_entry__.build()``).
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
SO = PKG / "libqasr_hip.so"
BINDING = PKG / "_binding.so"
ARCHIVE = PKG / "libqasr_hip.a"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))

ARCH = "gfx950"

# -ffp-contract=off keeps every a*b+c a separate multiply and add unless the
# source calls fmaf, so elementwise epilogues round exactly as written.
# Packed-fp32 instruction selection is disabled (v_pk_* f32 forms).
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]


def _hipcc() -> str:
    p = ROCM / "bin" / "hipcc"
    if p.exists():
        return str(p)
    found = shutil.which("hipcc")
    if not found:
        raise RuntimeError("hipcc not found; the gfx950 library cannot be built")
    return found


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}")


def _binding_includes() -> list[Path]:
    import torch

    t = Path(torch.__file__).resolve().parent
    return [t / "include", t / "include" / "torch" / "csrc" / "api" / "include", ROCM / "include",
            Path(sysconfig.get_paths()["include"])]


def binding_missing() -> str:
    """What keeps the Python binding from being built here ('' for nothing): it needs torch
    and its C++ headers, Python's headers and g++, which a C or Rust host has no use for."""
    try:
        incs = _binding_includes()
    except ImportError as e:
        return f"torch cannot be imported ({e})"
    for header in ("torch/csrc/autograd/python_variable.h", "c10/hip/HIPStream.h", "Python.h"):
        if not any((i / header).exists() for i in incs):
            return f"no {header}"
    return "" if shutil.which("g++") else "no g++"


def binding_command(out: Path) -> list[str]:
    """The compile line of the Python binding: plain host C++ that calls the
    entry points by address, so it links torch but not the kernel library."""
    import torch

    lib = Path(torch.__file__).resolve().parent / "lib"
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={abi}", *[f"-I{i}" for i in _binding_includes()], str(CSRC / "binding.cpp"),
            "-o", str(out), f"-L{lib}", "-ltorch_python", "-ltorch_cpu", "-lc10_hip", "-lc10"]


def build_binding(verbose: bool = False) -> Path | None:
    """Builds ``_binding.so``. Where its prerequisites are missing, says so and leaves none
    (an old one may not match the library): the libraries serve C and Rust hosts all the
    same, and ``kernels.py`` names the reason on its first call."""
    missing = binding_missing()
    if missing:
        print(f"the Python binding is not built: {missing}", file=sys.stderr, flush=True)
        BINDING.unlink(missing_ok=True)
        return None
    tmp = BUILD / "_binding.so"
    cmd = binding_command(tmp)
    if verbose:
        print(" ".join(cmd), flush=True)
    _run(cmd)
    os.replace(tmp, BINDING)
    return BINDING


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def build(verbose: bool = False) -> Path:
    """Compile all kernels and link the shared and static libraries; then the Python
    binding, where it can be built."""
    hipcc = _hipcc()
    BUILD.mkdir(exist_ok=True)
    srcs = sources()
    objs = [BUILD / (s.stem + ".o") for s in srcs]

    def compile_one(pair):
        src, obj = pair
        cmd = [hipcc, *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)

    workers = min(len(srcs), max(1, (os.cpu_count() or 4)))
    with ThreadPoolExecutor(max_workers=workers) as ex:
        binding = ex.submit(build_binding, verbose)  # beside the kernels; its outcome is looked at last
        list(ex.map(compile_one, zip(srcs, objs)))

    tmp_so = SO.with_suffix(".so.tmp")
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp_so),
          *map(str, objs)])
    os.replace(tmp_so, SO)

    if ARCHIVE.exists():
        ARCHIVE.unlink()
    _run(["ar", "rcs", str(ARCHIVE), *map(str, objs)])
    build_cpp_tests(hipcc, verbose)
    binding.result()
    return SO


ROOT = PKG.parent
CPP_TESTS = ROOT / "tests" / "cpp"
CPP_TEST_BIN = CPP_TESTS / "_build" / "test_kernels"


def build_cpp_tests(hipcc: str | None = None, verbose: bool = False) -> Path:
    """Builds the C++ host-mirror test against the static archive (so the
    binary carries its own copy of the kernels: the static-link path a Rust
    build.rs would use)."""
    hipcc = hipcc or _hipcc()
    CPP_TEST_BIN.parent.mkdir(exist_ok=True)
    obj = CPP_TEST_BIN.with_suffix(".o")
    tmp = CPP_TEST_BIN.with_suffix(".tmp")
    # compile and link separately: hipcc applies ``-x hip`` to every input
    # that follows a .cpp source, which would include the archive
    cmds = [[hipcc, f"--offload-arch={ARCH}", "-O2", "-std=c++17", "-Wall", "-I", str(ROOT / "include"),
             "-c", str(CPP_TESTS / "test_kernels.cpp"), "-o", str(obj)],
            [hipcc, f"--offload-arch={ARCH}", str(obj), str(ARCHIVE), "-o", str(tmp)]]
    for cmd in cmds:
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)
    os.replace(tmp, CPP_TEST_BIN)
    return CPP_TEST_BIN


if __name__ == "__main__":
    out = build(verbose="-v" in sys.argv)
    print(out)
