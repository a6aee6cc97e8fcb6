"""Build ``starter_amd/kernels/libqwen_fused.so`` from ``starter_amd/csrc/*.hip``.

Every source is compiled for gfx950 only, with:

* ``-ffp-contract=off`` - no silent multiply-add fusion; the kernels round to
  bf16 at exactly the points the reference does, and an FMA would change the
  f32 value being rounded;
* ``-Xclang -target-feature -Xclang -packed-fp32-ops`` - no packed-f32 VALU
  instructions (the host pass warns that it does not know the feature; that
  warning is harmless);
* HIP's default correctly rounded f32 divide and sqrt.

A second library, ``starter_amd/kernels/libqwen_fused_phases.so``, holds only
the decode attention built with ``-DQF_PHASE_STAMPS``: the same kernels plus
an instrumented entry point that records per-workgroup phase timestamps
(``starter_amd.attention_phases`` reads them).  Nothing in the product loads
it.

Run ``python -m starter_amd.build`` or call :func:`build`.
"""

from __future__ import annotations

import concurrent.futures
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PACKAGE = Path(__file__).resolve().parent
ROOT = PACKAGE.parent
CSRC = PACKAGE / "csrc"
OBJ_DIR = PACKAGE / "_build"
LIBRARY = PACKAGE / "kernels" / "libqwen_fused.so"
PHASES_LIBRARY = PACKAGE / "kernels" / "libqwen_fused_phases.so"
PHASES_SOURCE = "decode_attention.hip"
# one interpreter's ABI, by its name
HOST_CALLS = PACKAGE / "kernels" / f"_host_calls{sysconfig.get_config_var('EXT_SUFFIX')}"
HOST_SOURCE = "host_calls.cpp"
SOURCES = ("rmsnorm.hip", "silu_mul.hip", "qk_norm_rope.hip", "embedding.hip", "skinny_gemm.hip",
           "stream_gemm.hip", "decode_attention.hip", "prefill_attention.hip", "row_gemv.hip")
ARCH = "gfx950"

COMPILE_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-I", str(ROOT / "include"),
]
# Per-source additions.  The attention kernels rescale their f32
# accumulators between matrix-core products; with the accumulators in
# ordinary VGPRs (instead of AGPRs) no copies are needed between the two
# register files (prefill 1.3x, decode 2% faster, same occupancy).
_VGPR_MFMA = ["-mllvm", "-amdgpu-mfma-vgpr-form"]
EXTRA_FLAGS = {
    "decode_attention.hip": _VGPR_MFMA,
    "prefill_attention.hip": _VGPR_MFMA,
}


def hipcc() -> str:
    path = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError(f"hipcc not found (looked for {path})")
    return path


def _torch_dir() -> Path:
    return Path(importlib.util.find_spec("torch").origin).parent


def _cxx() -> str:
    return os.environ.get("CXX") or "g++"


def _host_flags() -> list[str]:
    """Flags of the Python extension: torch's and HIP's headers (HIP's want to
    know the platform when no HIP compiler says it), and the torch build they
    belong to, which the extension compares with the one that imports it."""
    from torch import version
    include = _torch_dir() / "include"
    return ["-O2", "-fPIC", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f'-DQF_TORCH_BUILD="{version.__version__} {version.git_version}"',
            "-I", str(ROOT / "include"), "-isystem", str(include),
            "-isystem", str(include / "torch" / "csrc" / "api" / "include"),
            "-isystem", str(Path(hipcc()).resolve().parents[1] / "include"),
            "-isystem", sysconfig.get_paths()["include"]]


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # The host pass always warns about the device-only packed-fp32 feature.
    noise = "'-packed-fp32-ops' is not a recognized feature"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)


def _compile_host(verbose: bool) -> Path:
    obj = OBJ_DIR / (Path(HOST_SOURCE).stem + ".o")
    _run([_cxx(), *_host_flags(), "-c", str(CSRC / HOST_SOURCE), "-o", str(obj)], verbose)
    return obj


def _link_host(obj: Path, verbose: bool) -> None:
    tmp = HOST_CALLS.with_suffix(".so.tmp")
    _run([_cxx(), "-shared", "-o", str(tmp), str(obj), f"-L{LIBRARY.parent}",
          f"-l:{LIBRARY.name}", "-Wl,-rpath,$ORIGIN", f"-L{_torch_dir() / 'lib'}", "-lc10", "-lc10_hip",
          "-ltorch_cpu", "-ltorch_python"], verbose)
    os.replace(tmp, HOST_CALLS)


def build(verbose: bool = False) -> Path:
    """Compile every HIP source and link the shared library (and the phase
    timing library), then the Python extension that calls it
    (``csrc/host_calls.cpp``, host code only); return the product library's
    path.  The extension is the only part that needs a host compiler and
    torch's headers; where it does not build, the library stands without it."""
    cc = hipcc()
    OBJ_DIR.mkdir(exist_ok=True)
    jobs = []
    for name in SOURCES:
        obj = OBJ_DIR / (Path(name).stem + ".o")
        jobs.append((obj, [cc, *COMPILE_FLAGS, *EXTRA_FLAGS.get(name, ()), "-c", str(CSRC / name),
                           "-o", str(obj)]))
    phases_obj = OBJ_DIR / (Path(PHASES_SOURCE).stem + "_phases.o")
    phases_job = (phases_obj, [cc, *COMPILE_FLAGS, *EXTRA_FLAGS.get(PHASES_SOURCE, ()),
                               "-DQF_PHASE_STAMPS", "-c", str(CSRC / PHASES_SOURCE),
                               "-o", str(phases_obj)])
    workers = min(len(jobs) + 2, max(1, min(8, os.cpu_count() or 1)))
    with concurrent.futures.ThreadPoolExecutor(workers) as pool:
        host_obj = pool.submit(_compile_host, verbose)
        for fut in [pool.submit(_run, cmd, verbose) for _, cmd in (*jobs, phases_job)]:
            fut.result()
    for library, objects in ((LIBRARY, [obj for obj, _ in jobs]), (PHASES_LIBRARY, [phases_obj])):
        tmp = library.with_suffix(".so.tmp")
        _run([cc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp),
              *[str(obj) for obj in objects]], verbose)
        os.replace(tmp, library)
    try:
        _link_host(host_obj.result(), verbose)
    except (RuntimeError, OSError, ImportError, AttributeError) as error:
        HOST_CALLS.unlink(missing_ok=True)  # never an older one beside a new library
        print(f"warning: {HOST_CALLS.name} is not built ({error}): kernel calls take the Python path, "
              "about 5 us more each", file=sys.stderr)
    return LIBRARY


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
