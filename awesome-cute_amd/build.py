"""Builds libmarlin_amd.so (HIP kernels + C ABI), _marlin_torch.so (the same calls on
tensors) and libmarlin_amd_probe.so (the measurement probes of the benchmark) in-tree
for gfx950."""
import importlib.util
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmarlin_amd.so")
BINDING = os.path.join(HERE, "_marlin_torch.so")
PROBE_LIB = os.path.join(HERE, "libmarlin_amd_probe.so")
# source -> extra flags.  The prefill kernel keeps its 128 accumulator registers
# in ordinary VGPRs (it fits in 256), which spares the AGPR copy traffic the
# default register split produces around every MFMA.
SOURCES = {
    "marlin_host.hip": [],
    "scratch_pool.hip": [],
    "w4a16_stream.hip": [],
    "w4a16_strip.hip": [],
    "w4a16_rows.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "w4a16_rows_wide.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "w4a16_prefill.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "w4a16_prefill_wide.hip": [],
    "w4a16_convert.hip": [],
    "f16_streamk.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "f16_tiles.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
}
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-I", os.path.join(HERE, "build"),
    # packed fp32 arithmetic stays off for every kernel in this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument",
]


# the tensor binding is host code over torch's headers, which name the platform
# through these two macros
CXX = os.environ.get("CXX", "g++")
TORCH = os.path.dirname(importlib.util.find_spec("torch").origin)
TORCH_LIBS = os.path.join(TORCH, "lib")
CXX_FLAGS = [
    "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
    "-I", os.path.join(TORCH, "include"), "-I", os.path.join(TORCH, "include/torch/csrc/api/include"),
    "-I", "/opt/rocm/include", "-I", sysconfig.get_paths()["include"],
]


def _compile_binding(objdir, verbose):
    obj = os.path.join(objdir, "torch_binding.o")
    _run([CXX] + CXX_FLAGS + ["-c", "-o", obj, os.path.join(CSRC, "torch_binding.cpp")], verbose)
    return obj


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed:\n{out}")
    if verbose and out.strip():
        print(out)


def build_library(verbose=False):
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    # the assembly statements of the four-wave kernels and of the rows kernel over 128
    # columns (prologue, main loop and accumulator hand-over with fixed registers) are
    # written by generators; the sources include them from the build directory
    for gen in ("gen_prefill_wide.py", "gen_rows_wide.py", "gen_dense.py"):
        _run([sys.executable, os.path.join(CSRC, gen), objdir], verbose)
    objs = [os.path.join(objdir, src.replace(".hip", ".o")) for src in SOURCES]
    with ThreadPoolExecutor(4) as pool:
        binding = pool.submit(_compile_binding, objdir, verbose)
        list(pool.map(lambda job: _run([HIPCC] + FLAGS + job[0][1] + ["-c", "-o", job[1],
                                                                      os.path.join(CSRC, job[0][0])],
                                       verbose), zip(SOURCES.items(), objs)))
        binding_obj = binding.result()
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs, verbose)
    _run([CXX, "-shared", "-o", BINDING, binding_obj, "-L", HERE, "-lmarlin_amd", "-L", TORCH_LIBS,
          "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"], verbose)
    # the probes: a library of their own that asks the first one for its plans
    obj = os.path.join(objdir, "w4a16_probe.o")
    _run([HIPCC] + FLAGS + ["-c", "-o", obj, os.path.join(CSRC, "w4a16_probe.hip")], verbose)
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", PROBE_LIB, obj, "-L", HERE,
          "-lmarlin_amd", "-Wl,-rpath,$ORIGIN"], verbose)
    return LIB


if __name__ == "__main__":
    print(build_library(verbose=True))
