"""Builds libretro_mi355.so (HIP kernels + host wave buffer) for gfx950, the C example over it and _step_calls.so (the calls of a
decode step from Python), all with hipcc.

    python -m retrievalattention_amd.build

The library is written next to this file so that it travels with the source tree.
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libretro_mi355.so")
HIP_SOURCES = ["capi.hip", "score.hip", "select.hip", "attend.hip", "gather.hip", "kmeans.hip", "lru.hip",
               "step.hip", "prefill.hip"]
CPP_SOURCES = ["wavebuf.cpp"]
ARCH = "gfx950"
# -ffp-contract=off: products and sums round separately unless the source says fmaf, which
# keeps the k-means reductions reproducible on a CPU.  The packed-fp32 feature is disabled
# because some of its instruction forms have been unreliable on this hardware.
# The first words of a kernel's arguments (fourteen at most, none of a struct) are in scalar registers when its waves
# start; a wave that loads them first waits a memory round trip before it can ask for anything else.  32 groups of 4
# heads, 8192 clusters: scoring + selection 26.1 -> 25.3 us, a step 45.3 -> 44.5.
HIP_FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-ffp-contract=off",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument",
             "-mllvm", "-amdgpu-kernarg-preload-count=16"]
# per-file additions: the k-means assignment reads every MFMA accumulator in its argmax
# epilogue, so its accumulators live in ordinary VGPRs (no accumulator-register copies)
EXTRA_HIP_FLAGS = {"kmeans.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}
CPP_FLAGS = ["-O3", "-std=c++17", "-fPIC", "-pthread"]


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError("build step failed: " + " ".join(cmd) + "\n" + r.stdout)
    return r.stdout


def build(verbose=False):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    jobs = []
    for s in HIP_SOURCES:
        o = os.path.join(objdir, s + ".o")
        jobs.append(([hipcc] + HIP_FLAGS + EXTRA_HIP_FLAGS.get(s, []) + ["-c", os.path.join(CSRC, s), "-o", o], o))
    for s in CPP_SOURCES:
        o = os.path.join(objdir, s + ".o")
        jobs.append(([hipcc] + CPP_FLAGS + ["-c", os.path.join(CSRC, s), "-o", o], o))
    with ThreadPoolExecutor(max_workers=min(6, len(jobs))) as ex:
        outs = list(ex.map(lambda j: _run(j[0]), jobs))
    if verbose:
        for o in outs:
            if o.strip():
                print(o)
    objs = [j[1] for j in jobs]
    _run([hipcc, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", LIB] + objs + ["-pthread"])
    build_capi_example(hipcc)
    _run(step_calls_command(hipcc))   # (last: it alone needs torch's headers)
    return LIB


# The Python calls of a decode step (csrc/step_calls.cpp): a module of its own, because it is bound to this interpreter and to
# torch, which the library is not.
STEP_CALLS = os.path.join(HERE, "_step_calls.so")


def step_calls_command(hipcc):
    import torch
    from torch.utils import cpp_extension
    include = [x for d in cpp_extension.include_paths("cuda") + [sysconfig.get_paths()["include"]] for x in ("-isystem", d)]
    libs = [f"-L{d}" for d in cpp_extension.library_paths("cuda") + [HERE]]
    return [hipcc, *CPP_FLAGS, "-Wall", "-shared", "-no-hip-rt", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", *include,
            os.path.join(CSRC, "step_calls.cpp"), "-o", STEP_CALLS, *libs, "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10",
            "-lc10_hip", "-l:libretro_mi355.so", "-Wl,-rpath,$ORIGIN"]


# A plain HIP program that drives a decode step through the C ABI (no Python, no torch); tests/test_gpu_capi.py
# runs it.  It finds the library next to the package through its run path.
CAPI_EXAMPLE_SRC = os.path.join(os.path.dirname(HERE), "tests", "capi_decode_step.cpp")
CAPI_EXAMPLE = os.path.join(os.path.dirname(HERE), "tests", "capi_decode_step")


def build_capi_example(hipcc):
    if not os.path.exists(CAPI_EXAMPLE_SRC):
        return None
    _run([hipcc, "-O2", "-std=c++17", f"--offload-arch={ARCH}", "-I", os.path.join(os.path.dirname(HERE), "include"),
          CAPI_EXAMPLE_SRC, "-o", CAPI_EXAMPLE, "-L", HERE, "-l:libretro_mi355.so",
          "-Wl,-rpath,$ORIGIN/../retrievalattention_amd"])
    return CAPI_EXAMPLE


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
