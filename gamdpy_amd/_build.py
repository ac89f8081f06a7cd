"""Build libgamdpy_amd.so for gfx950 with hipcc (in-tree, no JIT cache).

    python -m gamdpy_amd._build
"""
import concurrent.futures
import os
import shutil
import subprocess
import sys

_HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(_HERE)
# gmd_core.hip holds the host code and every kernel but the step kernels, which
# gmd_steps_inst.hip instantiates one (pair-function base, cutoff) group per
# compilation, and the NPT_Atomic kernels of each base in one more: the groups
# compile in parallel (the longest first) and are linked into one library
_CORE = os.path.join(_HERE, "csrc", "gmd_core.hip")
_INST = os.path.join(_HERE, "csrc", "gmd_steps_inst.hip")
SOURCES = [(_INST, f"steps_b{b}_c{c}", [f"-DGMD_INST_BASE={b}", f"-DGMD_INST_CUT={c}"])
           for b in (2, 3, 1) for c in range(3)] + \
          [(_INST, f"steps_b{b}_npt", [f"-DGMD_INST_BASE={b}", "-DGMD_INST_NPT"]) for b in (2, 3, 1, 0)] + \
          [(_INST, f"steps_b0_c{c}", ["-DGMD_INST_BASE=0", f"-DGMD_INST_CUT={c}"]) for c in range(3)] + \
          [(_CORE, "core", [])]
JOBS = max(1, min(8, os.cpu_count() or 1))   # compilations at a time
DEPS = [os.path.join(_HERE, "csrc", f) for f in ("gmd_device.h", "gmd_kernels.h", "gmd_steps.h", "gmd_adjoint.h")] + \
       [os.path.join(ROOT, "include", "gamdpy_amd.h")]
OUT = os.path.join(_HERE, "libgamdpy_amd.so")
# the reference's kernel design compiled for this GPU: a comparison point for
# the benchmark, a library of its own outside the product path
REF_SOURCE = os.path.join(_HERE, "csrc", "gmd_refdesign.hip")
REF_OUT = os.path.join(_HERE, "libgmd_refdesign.so")
ARCH = os.environ.get("GMD_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Wno-unused-result",
    # no packed FP32 instructions are generated (v_pk_*_f32)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc():
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build gamdpy_amd)")


def build(verbose=False):
    """Compile every HIP source (in parallel) and link gamdpy_amd/libgamdpy_amd.so
    (always recompiles)."""
    cc = hipcc()
    inc = ["-I", os.path.join(ROOT, "include")]
    jobs = [(src, OUT + "." + name + ".o", HIPCC_FLAGS + inc + defs + ["-c"]) for src, name, defs in SOURCES]
    jobs.append((REF_SOURCE, REF_OUT + ".tmp", HIPCC_FLAGS + ["-shared"]))
    failed = []

    def compile_one(job):
        src, out, flags = job
        cmd = [cc] + flags + [src, "-o", out]
        if verbose:
            print(" ".join(cmd), flush=True)
        res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        if res.returncode != 0:
            sys.stderr.write(res.stdout)
            failed.append(os.path.basename(out))

    with concurrent.futures.ThreadPoolExecutor(JOBS) as pool:
        list(pool.map(compile_one, jobs))
    if failed:
        raise RuntimeError(f"hipcc failed for {', '.join(failed)}")
    objs = [out for _, out, _ in jobs[:-1]]
    tmp = OUT + ".tmp"
    cmd = [cc, f"--offload-arch={ARCH}", "-shared", "-fPIC"] + objs + ["-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError(f"hipcc link failed with exit code {res.returncode}")
    for obj in objs:
        os.remove(obj)
    os.replace(REF_OUT + ".tmp", REF_OUT)
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
