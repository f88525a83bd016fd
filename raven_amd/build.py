"""Builds ``raven_amd/csrc/libnxhip.so`` for gfx950 with hipcc.

One object per ``.hip`` translation unit (compiled in parallel), linked into a
single shared library that exports exactly the C ABI of ``include/nxhip.h``; and
the Python module of its host path, with gcc.
Cross-compiles without a GPU.
"""

from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

CSRC = Path(__file__).resolve().parent / "csrc"
OBJ = CSRC / "build"
LIB = CSRC / "libnxhip.so"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    # mul and add stay separate roundings wherever the source says so
    "-ffp-contract=off",
    # no packed-FP32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-value", "-Wno-unused-function",
]


# Extra flags of single sources. attention.hip: the output accumulators are both MFMA
# results and operands of vector instructions (the rescale by e^(old max - new max)); with
# the compiler's default they live in AGPRs and are copied to VGPRs and back in every key
# tile (288 v_accvgpr moves in the loop, 214 registers, 2 waves per SIMD). Asking for the
# VGPR form of MFMA removes the copies: 152 registers, 3 waves per SIMD.
PER_SOURCE_FLAGS = {
    "attention.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
}


def sources():
    return sorted(CSRC.glob("*.hip"))


def _stale(src: Path, obj: Path) -> bool:
    if not obj.exists():
        return True
    newest = max(p.stat().st_mtime for p in [src, *CSRC.glob("*.hpp"),
                                             CSRC.parent.parent / "include" / "nxhip.h"])
    return obj.stat().st_mtime < newest


def _compile(src: Path, force: bool) -> Path:
    obj = OBJ / (src.stem + ".o")
    if force or _stale(src, obj):
        cmd = [HIPCC, *FLAGS, *PER_SOURCE_FLAGS.get(src.name, []), "-c", str(src), "-o", str(obj)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src.name}:\n{err}")
        if err.strip():
            print(err, file=sys.stderr)
    return obj


def build_all(force: bool = True, jobs: int | None = None) -> Path:
    OBJ.mkdir(exist_ok=True)
    jobs = jobs or min(8, os.cpu_count() or 1)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, force), sources()))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(LIB), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    build_calls()
    return LIB


CALLS_SRC = CSRC.parent / "host_c" / "nx_calls.c"
CALLS_LIB = CSRC.parent / ("_nxcalls" + sysconfig.get_config_var("EXT_SUFFIX"))  # found by this Python's ABI only


def build_calls() -> Path:
    """The Python module of the per-primitive host path (raven_amd/host_c/nx_calls.c): gcc only."""
    cmd = ["gcc", "-std=gnu11", "-O2", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-Wextra",
           "-I", str(CSRC.parent.parent / "include"), "-I", sysconfig.get_paths()["include"],
           "-o", str(CALLS_LIB), str(CALLS_SRC)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0 or r.stderr.strip():
        raise RuntimeError(f"gcc failed on {CALLS_SRC.name}:\n{r.stderr}")
    return CALLS_LIB


ABI_CHECK_SRC = CSRC.parent.parent / "tests" / "abi_c" / "nxh_abi_check.c"
ABI_CHECK_BIN = ABI_CHECK_SRC.with_suffix("")


def build_abi_check() -> Path:
    """The plain-C user of the ABI (tests/abi_c): gcc, no HIP, no Python at run time."""
    cmd = ["gcc", "-std=gnu11", "-O1", "-Wall", "-Wextra", "-I", str(CSRC.parent.parent / "include"),
           "-o", str(ABI_CHECK_BIN), str(ABI_CHECK_SRC), "-ldl", "-lm"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0 or r.stderr.strip():
        raise RuntimeError(f"gcc failed on {ABI_CHECK_SRC.name}:\n{r.stderr}")
    return ABI_CHECK_BIN


GPT2_HOST_SRC = CSRC.parent / "host_c" / "kaun_gpt2_host.c"
GPT2_HOST_BIN = GPT2_HOST_SRC.with_suffix("")


def build_gpt2_host() -> Path:
    """The compiled host of Kaun's GPT-2 forward over the C ABI (raven_amd/host_c): gcc only."""
    cmd = ["gcc", "-std=gnu11", "-O2", "-Wall", "-Wextra", "-I", str(CSRC.parent.parent / "include"),
           "-o", str(GPT2_HOST_BIN), str(GPT2_HOST_SRC), "-ldl", "-lm"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0 or r.stderr.strip():
        raise RuntimeError(f"gcc failed on {GPT2_HOST_SRC.name}:\n{r.stderr}")
    return GPT2_HOST_BIN


MFMA_PROBE_SRC = CSRC.parent.parent / "bench_mfma_probe.hip"
MFMA_PROBE_LIB = MFMA_PROBE_SRC.with_suffix(".so")


def build_mfma_probe() -> Path:
    """The MFMA-only loop bench.py --gemm-study times beside the GEMMs (not part of libnxhip)."""
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", str(MFMA_PROBE_SRC), "-o", str(MFMA_PROBE_LIB)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {MFMA_PROBE_SRC.name}:\n{r.stderr}")
    return MFMA_PROBE_LIB


if __name__ == "__main__":
    print(build_all(force="--force" in sys.argv))
