"""Build liblighthouse_hip.so (gfx950).

Usage: ``python -m lighthouse_amd.build`` or ``lighthouse_amd.build.build_hip()``.
hipcc cross-compiles for gfx950 without a GPU present.  Objects go to ``build/``,
the libraries to ``lighthouse_amd/lib/`` (all git-ignored).
"""

from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "lighthouse_amd" / "csrc"
LIB_DIR = ROOT / "lighthouse_amd" / "lib"
LIB_PATH = LIB_DIR / "liblighthouse_hip.so"
PROBE_LIB = LIB_DIR / "liblighthouse_probe.so"  # bench.py's MFMA-rate probe, not part of the product library

HIP_SOURCES = ["runtime.hip", "gemm16.hip", "gemm16_direct.hip", "gemm32.hip", "gemm8.hip", "gemm_small.hip", "gemm_small_norm.hip", "attention.hip", "attention_small.hip", "rowwise.hip", "api.hip"]

# A lone workgroup's main loop fetches a line more of instructions a turn where it starts at the end of one: the same loop 4 bytes
# before a multiple of 64 and on it, 2923 x 768 x 5824 bf16 41.7 and 40.6 us.
ALIGNED_LOOPS = ["-falign-loops=64"]

# Sources compiled more than once, with different macros: {source: {suffix of the object: macros and flags}}.
INSTANCES = {
    "gemm16_direct.hip": {
        f"_{dt}_{tm}{tn}{'_large' * large}": [f"-DLH_GEMM16_DT=LH_{dt.upper()}", f"-DLH_GEMM16_TM={tm}", f"-DLH_GEMM16_TN={tn}",
                                             f"-DLH_GEMM16_LARGE={large}"] + ALIGNED_LOOPS * (tm == 0)
        for tm, tn, large in ((4, 2, 1), (4, 2, 0), (4, 1, 0), (2, 2, 0), (2, 1, 0), (0, 0, 0)) for dt in ("bf16", "f16")
    } | {
        f"_{dt}_{kind}_{tm}{tn}": [f"-DLH_GEMM16_DT=LH_{dt.upper()}", f"-DLH_GEMM16_TM={tm}", f"-DLH_GEMM16_TN={tn}", "-DLH_GEMM16_LARGE=0",
                                   f"-DLH_GEMM16_{kind.upper()}=1"] + ALIGNED_LOOPS * (kind == "deep")
        for kind, tm, tn in (("odd", 2, 1), ("deep", 2, 1), ("deep", 2, 3), ("deep", 2, 2), ("deep", 4, 1)) for dt in ("bf16", "f16")
    },
}

HIPCC_FLAGS = [
    "-O3",
    "--offload-arch=gfx950",
    "-std=c++17",
    "-fPIC",
    # Packed FP32 instructions are kept out of the generated code on purpose.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{ROOT / 'include'}",
    f"-I{CSRC}",
]


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout)
        sys.stderr.write(proc.stderr)
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}")


def build_hip(verbose: bool = False) -> Path:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    obj_dir = ROOT / "build" / "obj"
    obj_dir.mkdir(parents=True, exist_ok=True)
    LIB_DIR.mkdir(parents=True, exist_ok=True)

    def compile_one(src: str, suffix: str = "", macros: tuple = ()) -> str:
        obj = obj_dir / (Path(src).stem + suffix + ".o")
        cmd = [hipcc, *HIPCC_FLAGS, *macros, "-c", str(CSRC / src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)
        return str(obj)

    jobs = [(src, suffix, macros) for src, many in INSTANCES.items() for suffix, macros in many.items()]
    jobs += [(src, "", ()) for src in HIP_SOURCES if src not in INSTANCES]
    with ThreadPoolExecutor(max_workers=8) as pool:
        probe = pool.submit(compile_one, "probe.hip")
        objs = list(pool.map(lambda job: compile_one(*job), jobs))
        probe_obj = probe.result()
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", str(LIB_PATH)])
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", probe_obj, "-o", str(PROBE_LIB)])
    return LIB_PATH


if __name__ == "__main__":
    print(f"built {build_hip(verbose=True)}")
