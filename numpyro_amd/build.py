"""Builds libnumpyro_amd.so for gfx950 in-tree with hipcc.

Each translation unit compiles to its own object (in parallel, objects under
numpyro_amd/_build/), then one hipcc line links the shared library.  The
units share host-level interfaces only (nax_internal.h), so no relocatable
device code is needed."""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
OUT = os.path.join(HERE, "libnumpyro_amd.so")
SOURCES = ["sampler.hip", "logistic.hip", "logistic_mfma.hip", "logistic_split.hip",
           "logistic_rows.hip", "logistic_chain.hip", "sv.hip", "hier.hip", "diagnostics.hip", "ecs.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # packed FP32 instructions stay off (v_pk_{add,mul,fma}_f32)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]
# logistic_split: its wide kernels use more than 256 registers and add to their
# accumulators outside the MFMAs; left to itself the compiler keeps those in the
# accumulation registers and copies them out and back around every addition
# (500,000 x 250, 250 chains, fp8: 1024 us, 948 with the flag; fp32: 928 and 853)
FILE_FLAGS = {"logistic_split.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def _run(cmd, what):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"hipcc failed: {what}")
    return r


def build(verbose=False, jobs=None):
    os.makedirs(OBJ, exist_ok=True)
    objs = [os.path.join(OBJ, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    cmds = [[HIPCC] + FLAGS + FILE_FLAGS.get(s, []) + ["-c", os.path.join(CSRC, s), "-o", o]
            for s, o in zip(SOURCES, objs)]
    if verbose:
        for c in cmds:
            print(" ".join(c), flush=True)
    jobs = jobs or min(len(cmds), os.cpu_count() or 1)
    with ThreadPoolExecutor(jobs) as ex:
        list(ex.map(lambda c: _run(c, c[-3]), cmds))
    tmp = OUT + ".tmp"
    link = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", tmp]
    if verbose:
        print(" ".join(link), flush=True)
    _run(link, "link libnumpyro_amd.so")
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
