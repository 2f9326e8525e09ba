"""Builds the native libraries of litert_amd for gfx950 with hipcc, in-tree.

    python -m litert_amd.build            # everything
    python -m litert_amd.build --only fc  # just the kernel library

Outputs land in litert_amd/lib/ (git-ignored; they travel to the GPU box with the tree).
"""
import argparse
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.environ.get("LITERT_AMD_LIB_DIR", os.path.join(HERE, "lib"))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# -ffp-contract=off: several float steps reproduce the reference's unfused
# multiply-then-add; packed-fp32 ops are disabled (some of their forms have given wrong results).
COMMON = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wall",
          "-Wno-unused-function", "-I" + os.path.join(ROOT, "include")]
# Kernel-argument preloading (gfx940 and later): the leading scalar arguments of a kernel
# arrive in registers with the wavefront instead of through a first round of scalar loads.
COMMON += ["-mllvm", "-amdgpu-kernarg-preload-count=16"]
COMMON += os.environ.get("LITERT_AMD_EXTRA_HIPCC_FLAGS", "").split()

FC_SOURCES = ["capi.hip", "quantize.hip", "fc_int8_gemv.hip", "fc_int8_packed_gemv.hip", "fc_int8_rows_gemv.hip", "fc_int8_packed_gemm.hip", "fc_int8_split_gemm.hip",
              "fc_int8_gemm_mfma.hip", "fc_int4_blockwise.hip", "fc_int4_packed.hip", "fc_int4_per_channel_gemv.hip",
              "embedding_lookup.hip", "fc_int4_blockwise_gemm.hip"]


def _run(cmd):
    print("+", " ".join(cmd), flush=True)
    subprocess.check_call(cmd)


# Per-file additions. The blockwise int4 GEMM reads every MFMA result with the vector ALU right
# away (one MFMA per quantization block), so its results should land in ordinary vector
# registers: with the default choice of accumulation registers each of them costs a copy
# instruction first (a quarter of the kernel's vector work).
FILE_FLAGS = {"fc_int4_blockwise_gemm.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def build_fc():
    os.makedirs(LIB, exist_ok=True)
    objs = []
    procs = []
    for src in FC_SOURCES:
        obj = os.path.join(LIB, src.replace(".hip", ".o"))
        cmd = [HIPCC] + COMMON + FILE_FLAGS.get(src, []) + ["-c", os.path.join(CSRC, src), "-o", obj]
        print("+", " ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd)))
        objs.append(obj)
    for src, p in procs:
        if p.wait() != 0:
            raise RuntimeError("hipcc failed on " + src)
    out = os.path.join(LIB, "liblitert_amd_fc.so")
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out] + objs)
    return out


def build_python_calls():
    """The per-call entry points as a CPython extension (host code only), named for the interpreter it
    is built for. Without that interpreter's headers there is none, and the ops use ctypes."""
    include = sysconfig.get_paths()["include"]
    if not os.path.exists(os.path.join(include, "Python.h")):
        print("no Python.h in %s: litert_amd_calls is not built" % include, flush=True)
        return None
    out = os.path.join(LIB, "litert_amd_calls" + sysconfig.get_config_var("EXT_SUFFIX"))
    _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
          "-I" + os.path.join(ROOT, "include"), "-I" + include, "-o", out,
          os.path.join(CSRC, "host", "python_calls.cc"), "-L" + LIB, "-llitert_amd_fc",
          "-Wl,-rpath,$ORIGIN"])
    return out


def torch_tensors_name(torch_version):
    """File name of the extension that allocates output tensors: it is bound to one torch and one
    interpreter."""
    tag = "".join(c if c.isalnum() else "_" for c in torch_version)
    return "litert_amd_tensors-torch" + tag + sysconfig.get_config_var("EXT_SUFFIX")


def build_torch_tensors():
    """Output tensors and scratch for the Python ops without torch.empty's argument parsing (host code
    only). Without torch or the interpreter's headers, or where they do not compile, there is none, and the
    ops use torch.empty; nothing else needs it."""
    try:
        import torch
    except (ImportError, OSError) as e:
        print("no torch (%s): litert_amd_tensors is not built" % e, flush=True)
        return None
    root = os.path.dirname(torch.__file__)
    python = sysconfig.get_paths()["include"]
    if not (os.path.exists(os.path.join(python, "Python.h")) and
            os.path.exists(os.path.join(root, "include", "ATen", "ATen.h"))):
        print("no headers of torch or Python: litert_amd_tensors is not built", flush=True)
        return None
    out = os.path.join(LIB, torch_tensors_name(torch.__version__))
    try:
        _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-w",
              "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
              "-I" + os.path.join(root, "include"),
              "-I" + os.path.join(root, "include", "torch", "csrc", "api", "include"), "-I" + python,
              "-o", out, os.path.join(CSRC, "host", "torch_tensors.cc"), "-L" + os.path.join(root, "lib"),
              "-lc10", "-ltorch_cpu", "-ltorch_python"])
    except (subprocess.CalledProcessError, OSError) as e:
        print("%s: litert_amd_tensors is not built" % e, flush=True)
        if os.path.exists(out):
            os.remove(out)  # an earlier build's, which the ops would load
        return None
    return out


def build_delegate():
    src_dir = os.path.join(CSRC, "delegate")
    if not os.path.isdir(src_dir):
        return None
    srcs = sorted(os.path.join(src_dir, f) for f in os.listdir(src_dir) if f.endswith(".cc"))
    if not srcs:
        return None
    out = os.path.join(LIB, "liblitert_amd_delegate.so")
    _run([HIPCC, "-x", "hip"] + COMMON + ["-shared", "-o", out] + srcs +
         ["-L" + LIB, "-llitert_amd_fc", "-Wl,-rpath,$ORIGIN"])
    return out


def build_bench_probes():
    """The benchmark's measurement aids: a library of their own, not linked into the others."""
    os.makedirs(LIB, exist_ok=True)
    out = os.path.join(LIB, "liblitert_amd_bench_probes.so")
    _run([HIPCC] + COMMON + ["-shared", "-o", out, os.path.join(HERE, "bench_probes", "probes.hip")])
    return out


def build_all():
    outs = [build_fc(), build_python_calls(), build_bench_probes(), build_delegate(),
            build_torch_tensors()]
    return [out for out in outs if out]


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--only", choices=["fc", "delegate", "probes"])
    args = ap.parse_args()
    if args.only == "fc":
        build_fc()
        build_python_calls()
        build_torch_tensors()
    elif args.only == "delegate":
        build_delegate()
    elif args.only == "probes":
        build_bench_probes()
    else:
        build_all()
    sys.exit(0)
