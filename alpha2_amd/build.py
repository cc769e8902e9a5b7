"""Builds libalpha_hip.so for gfx950 from alpha2_amd/csrc/*.hip with hipcc (cross-compiles without a GPU).

    python -m alpha2_amd.build [--force]
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIB_DIR, "libalpha_hip.so")
SOURCES = ["runtime", "elementwise", "reduce", "nn", "optimizer", "gemm", "gemm_f32", "gemm_bf16", "gemm_bf16_dma_nt", "gemm_bf16_dma_nn",
           "gemm_bf16_dma_tn", "attention", "attention_bf16", "decode", "probe"]
# -packed-fp32-ops off: the compiler must not form v_pk_*_f32 from ordinary float code on this target.
FLAGS = ["--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-command-line-argument"]


def _hipcc() -> str:
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if c and (os.path.isabs(c) and os.path.exists(c) or not os.path.isabs(c)):
            return c
    return "hipcc"


def _compile(name: str, force: bool) -> str:
    src = os.path.join(CSRC, name + ".hip")
    obj = os.path.join(OBJ, name + ".o")
    deps = [src, os.path.join(CSRC, "common.h"), os.path.join(CSRC, "gemm_common.h"), os.path.join(CSRC, "gemm_bf16_dma.inc"),
            os.path.join(CSRC, "attention_common.h"), os.path.join(CSRC, "split_bf16.h"), os.path.join(CSRC, "dropout.h"), os.path.join(HERE, "..", "include", "alpha_hip.h")]
    if not force and os.path.exists(obj) and all(os.path.getmtime(obj) >= os.path.getmtime(d) for d in deps):
        return obj
    cmd = [_hipcc()] + FLAGS + ["-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {name}.hip:\n{r.stderr}")
    return obj


def build(force: bool = False, jobs: int = 8) -> str:
    os.makedirs(OBJ, exist_ok=True)
    os.makedirs(LIB_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda n: _compile(n, force), SOURCES))
    if force or not os.path.exists(LIB) or any(os.path.getmtime(o) > os.path.getmtime(LIB) for o in objs):
        r = subprocess.run([_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stderr}")
    return LIB


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
