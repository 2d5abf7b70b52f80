"""Ahead-of-time build of the HIP library (``libflashim_amd.so``, gfx950) and of the host build of its scalar numerics
(``libfim_host.so``, used by the CPU tests), and the device probes the tests and the bench use
(``libflashim_amd_probe.so``: numerics hooks and an MFMA microbenchmark, kept out of the product library), and the torch
operators on top of the C ABI (``libflashim_amd_torch.so``). The libraries are built in-tree so they travel with the
source tree; the loaders in :mod:`flashim_amd._lib` and :mod:`flashim_amd.library` only load what is built and never
compile at import time.

Flags: ``-ffp-contract=off`` keeps the epilogues' separate multiply and add roundings (the reference's order) unless a
kernel asks for an FMA explicitly; ``-packed-fp32-ops`` is disabled for all device code.
"""

from __future__ import annotations

import os
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PACKAGE = Path(__file__).resolve().parent
CSRC = PACKAGE / "csrc"
BUILD = PACKAGE / "_build"
LIBRARY = PACKAGE / "libflashim_amd.so"
HOST_LIBRARY = PACKAGE / "libfim_host.so"
DEVICE_SOURCES = (
    "quantize.hip", "igemm.hip", "deep_plan.hip", "deep_int8.hip", "deep_mx.hip", "depthwise.hip", "dwpw.hip", "mlp.hip",
    "stem.hip", "pointwise.hip", "version.hip",
)
PROBE_LIBRARY = PACKAGE / "libflashim_amd_probe.so"
PROBE_SOURCES = ("probe.hip", "deep_plan.hip")
TORCH_LIBRARY = PACKAGE / "libflashim_amd_torch.so"
ARCH = os.environ.get("FLASHIM_AMD_ARCH", "gfx950")
HIP_FLAGS = (
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-ffp-contract=off", "-munsafe-fp-atomics",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", f"-I{CSRC}",
)


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found: the flashim_amd HIP library cannot be built")
    return path


def _run(cmd: list[str]) -> None:
    result = subprocess.run(cmd, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"build step failed ({' '.join(cmd)}):\n{result.stderr[-4000:]}")


def build_torch_ops() -> Path:
    """Compile ``csrc/torch_ops.cpp`` against the installed torch and link it to ``libflashim_amd.so`` beside it (Python's
    own symbols come from the interpreter that loads it)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    temporary = TORCH_LIBRARY.with_suffix(f".{os.getpid()}.tmp")
    torch_lib = Path(torch.__file__).parent / "lib"
    includes = [flag for path in (*cpp_extension.include_paths("cuda"), sysconfig.get_path("include"))
                for flag in ("-isystem", path)]
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *includes, str(CSRC / "torch_ops.cpp"),
          "-o", str(temporary), f"-L{PACKAGE}", "-lflashim_amd", f"-L{torch_lib}", "-lc10", "-ltorch_cpu", "-lc10_hip",
          "-Wl,-rpath,$ORIGIN"])
    temporary.replace(TORCH_LIBRARY)
    return TORCH_LIBRARY


def build(jobs: int = 6) -> Path:
    """Compile every HIP source for gfx950 and link ``libflashim_amd.so``; build the torch operators on it and
    ``libfim_host.so``. Always rebuilds."""
    BUILD.mkdir(exist_ok=True)
    compiler = hipcc()
    sources = tuple(dict.fromkeys(DEVICE_SOURCES + PROBE_SOURCES))
    objects = {src: BUILD / (src.rsplit(".", 1)[0] + ".o") for src in sources}
    commands = [[compiler, *HIP_FLAGS, "-c", str(CSRC / src), "-o", str(objects[src])] for src in sources]
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        list(pool.map(_run, commands))
    for library, srcs in ((LIBRARY, DEVICE_SOURCES), (PROBE_LIBRARY, PROBE_SOURCES)):
        temporary = library.with_suffix(f".{os.getpid()}.tmp")
        _run([compiler, "-shared", "-fPIC", f"--offload-arch={ARCH}", *(str(objects[s]) for s in srcs),
              "-o", str(temporary)])
        temporary.replace(library)
    build_torch_ops()
    host_tmp = HOST_LIBRARY.with_suffix(f".{os.getpid()}.tmp")
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", str(CSRC / "numerics_host.cpp"), "-o", str(host_tmp)])
    host_tmp.replace(HOST_LIBRARY)
    return LIBRARY


if __name__ == "__main__":
    print(build())
