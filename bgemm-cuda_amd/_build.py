"""Builds libbgemm_mi355x.so for gfx950 with hipcc (no torch extension machinery), and _bgemm_native.so, the host side of the
layers on torch's C++ API, with the host compiler."""
import importlib.util
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
SO = os.path.join(HERE, "libbgemm_mi355x.so")
NATIVE_SO = os.path.join(HERE, "_bgemm_native.so")
SOURCES = ["api.hip", "pack.hip", "gemm_mfma.hip", "gemm_valu.hip", "gemm_skinny.hip", "gemm_chain.hip", "linear_rows.hip", "train.hip", "attention.hip", "attention_products.hip", "attention_grad.hip"]
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
         # "#pragma unroll" on loops with run-time bounds is a request, not a requirement
         "-Wno-pass-failed",
         # keep the compiler from forming packed-fp32 VALU ops
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def native_command():
    """The host compiler's command for _bgemm_native.so (torch is located, not imported).  NDEBUG, as torch itself is built: pybind11's
    debug counter would give the library a TLS segment.  One that is loaded after torch and never touched leaves every access to
    torch's own thread-local variables on the slow path of glibc's __tls_get_addr: an attention block of small kernels took
    291 us instead of 262, a packed product 9.7 instead of 8.8."""
    torch_dir = importlib.util.find_spec("torch").submodule_search_locations[0]
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return [os.environ.get("CXX", "g++"), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
            "-I" + os.path.join(torch_dir, "include"), "-I" + os.path.join(torch_dir, "include", "torch", "csrc", "api", "include"),
            "-I" + os.path.join(rocm, "include"), "-I" + sysconfig.get_paths()["include"], os.path.join(CSRC, "torch_ops.cpp"), os.path.join(CSRC, "torch_infer.cpp"), "-o", NATIVE_SO,
            "-L" + os.path.join(torch_dir, "lib"), "-lc10", "-ltorch_cpu", "-ltorch_python", "-lc10_hip", "-L" + HERE, "-l:" + os.path.basename(SO),
            "-Wl,-rpath,$ORIGIN"]


def build(verbose=True):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objs = []
    procs = []
    os.makedirs(os.path.join(HERE, "build"), exist_ok=True)
    for s in SOURCES:
        o = os.path.join(HERE, "build", s.replace(".hip", ".o"))
        objs.append(o)
        cmd = [hipcc] + FLAGS + ["-c", os.path.join(CSRC, s), "-o", o]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((s, subprocess.Popen(cmd)))
    for s, p in procs:
        if p.wait() != 0:
            raise RuntimeError("hipcc failed on %s" % s)
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", SO] + objs
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    cmd = native_command()
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return SO


def build_probes(root, verbose=True):
    """bench.py's measurement probes (bench_probes.hip beside it) -> libbench_probes.so, not part of the library."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    so = os.path.join(root, "libbench_probes.so")
    cmd = [hipcc] + FLAGS + ["-shared", "-o", so, os.path.join(root, "bench_probes.hip")]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return so


if __name__ == "__main__":
    build()
    sys.stdout.write(SO + "\n")
