"""Build libpie_hip.so (the gfx950 kernels + C ABI) in-tree with hipcc.

    python -m pie_amd.build          # or: python pie_amd/build.py

Each ``csrc/*.hip`` file is compiled in parallel to ``pie_amd/_build/*.o`` and linked into
``pie_amd/libpie_hip.so``. hipcc cross-compiles for gfx950 without a GPU present.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import warnings
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "libpie_hip.so"
# measurement probes (plain kernels with a hot-path kernel's access pattern; bench.py --op ceiling)
PROBE_SRC = PKG / "probe" / "probe.hip"
PROBE_LIB = PKG / "libpie_probe.so"
# the native call path of the small ops (a CPython module on torch's C++ API, host code only)
FAST_SRC = CSRC / "host" / "fast.cpp"
FAST_LIB = PKG / "_fast.so"
ARCH = "gfx950"

# Packed fp32 VALU ops are disabled: hipcc would otherwise form v_pk_{add,mul,fma}_f32 from
# ordinary float code, and some of their forms are unreliable on the target machines.
HIP_FLAGS = [
    "-O3",
    "-std=c++17",
    "-fPIC",
    f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (needs ROCm)")


def _compile(hipcc: str, src: Path, build_dir: Path, defines: tuple[str, ...]) -> Path:
    obj = build_dir / (src.stem + ".o")
    cmd = [hipcc, *HIP_FLAGS, *[f"-D{d}" for d in defines], "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{res.stdout}\n{res.stderr}")
    return obj


def build(verbose: bool = False, out: Path | None = None, defines: tuple[str, ...] = ()) -> Path:
    """Compile every kernel source and link libpie_hip.so (or ``out``); returns its path.
    ``defines`` (e.g. ``("PIE_NT_LOAD=0",)``) produce measurement variants of the library."""
    hipcc = _hipcc()
    lib = Path(out) if out else LIB
    build_dir = BUILD if not defines else BUILD / ("v_" + "_".join(defines).replace("=", ""))
    build_dir.mkdir(parents=True, exist_ok=True)
    fast = None
    if not defines and out is None:
        pool = cf.ThreadPoolExecutor(max_workers=1)
        fast = pool.submit(_try_build_fast, verbose)  # beside the kernels
        pool.shutdown(wait=False)
    srcs = sorted(CSRC.glob("*.hip"))
    if not srcs:
        raise RuntimeError(f"no kernel sources under {CSRC}")
    jobs = min(len(srcs), int(os.environ.get("MAX_JOBS", "8")), 16)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(hipcc, s, build_dir, tuple(defines)), srcs))
    tmp = lib.with_suffix(".so.tmp")
    cmd = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, lib)
    if verbose:
        print(f"built {lib}")
    if fast is not None:
        build_probe(verbose)
        fast.result()
    return lib


def _try_build_fast(verbose: bool) -> None:
    """build_fast, which the kernels and the C ABI do without: a failure leaves no module and warns."""
    try:
        build_fast(verbose)
    except (RuntimeError, ImportError, OSError) as e:
        FAST_LIB.unlink(missing_ok=True)
        warnings.warn(f"pie_amd: the native call path was not built, small ops take the slower general path: {e}",
                      RuntimeWarning, stacklevel=2)


def build_fast(verbose: bool = False) -> Path:
    """The native call path, against the installed torch's headers and libraries."""
    import sysconfig

    import torch

    root = Path(torch.__file__).parent
    rocm = Path(_hipcc()).resolve().parents[1]
    tmp = FAST_LIB.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-w",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           *[f"-I{p}" for p in (root / "include", root / "include/torch/csrc/api/include",
                                rocm / "include", sysconfig.get_paths()["include"])],
           str(FAST_SRC), f"-L{root / 'lib'}", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip",
           "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for {FAST_SRC.name}:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, FAST_LIB)
    if verbose:
        print(f"built {FAST_LIB}")
    return FAST_LIB


def build_probe(verbose: bool = False) -> Path:
    """The measurement-probe library (not part of the C ABI)."""
    tmp = PROBE_LIB.with_suffix(".so.tmp")
    cmd = [_hipcc(), *HIP_FLAGS, "-shared", "-o", str(tmp), str(PROBE_SRC)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {PROBE_SRC.name}:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, PROBE_LIB)
    if verbose:
        print(f"built {PROBE_LIB}")
    return PROBE_LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
