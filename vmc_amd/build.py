"""Builds the HIP library vmc_amd/libvmc_afqmc.so for gfx950 (in-tree), and the
host test programs that use it through include/vmc_afqmc.hpp.

    python -m vmc_amd.build            # compile changed sources, link
    python -m vmc_amd.build --force    # recompile everything

Every HIP source is compiled with hipcc --offload-arch=gfx950 and with packed
FP32 instructions disabled (-Xclang -target-feature -Xclang -packed-fp32-ops).
"""
import argparse
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libvmc_afqmc.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
SOURCES = ["afq_kernels.hip", "afq_force_bias.hip", "afq_prop64.hip", "afq_exchange64.hip", "afq_green.hip", "afq_qr.hip", "afq_vhs64.hip", "afq_exchange_pw2.hip", "afq_exchange_pw2x3.hip", "afq_mlp.hip", "afq_ctx.cpp", "afq_driver.cpp",
           "afq_noalloc.cpp"]
# per-file hipcc options: the pair-wise exchange keeps its MFMA accumulators in VGPRs
SOURCE_FLAGS = {"afq_exchange_pw2.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}
HEADERS = ["afq_device.hpp", "afq_internal.hpp", "afq_group.hpp", "afq_exchange_pw2.hpp", "afq_gemm64.hpp"]
CPP_TESTS = [("tests/cpp/api_parity.cpp", "tests/cpp/api_parity")]  # host programs over the C++ mirror
# FCIDUMP_chol (HDF5) reader/writer, a host library of its own: built where the HDF5 C
# library is installed (HDF5_DIR, default /opt/conda), skipped otherwise
HDF5_DIR = os.environ.get("HDF5_DIR", "/opt/conda")
IO_SRC = os.path.join(CSRC, "afq_fcidump.cpp")
IO_LIB = os.path.join(HERE, "libvmc_fcidump.so")
FLAGS = ["--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-Wall",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-I" + os.path.join(ROOT, "include")]


def _deps_mtime():
    paths = [os.path.join(CSRC, h) for h in HEADERS if os.path.exists(os.path.join(CSRC, h))]
    paths.append(os.path.join(ROOT, "include", "vmc_afqmc.h"))
    return max(os.path.getmtime(p) for p in paths)


def build(force=False, verbose=True):
    os.makedirs(OBJ, exist_ok=True)
    objs = []
    hdr_t = _deps_mtime()
    for src in SOURCES:
        sp = os.path.join(CSRC, src)
        if not os.path.exists(sp):
            continue
        op = os.path.join(OBJ, src + ".o")
        objs.append(op)
        if (not force and os.path.exists(op) and os.path.getmtime(op) > os.path.getmtime(sp)
                and os.path.getmtime(op) > hdr_t):
            continue
        cmd = ([HIPCC] + FLAGS + SOURCE_FLAGS.get(src, []) + (["-x", "hip"] if src.endswith(".cpp") else [])
               + ["-c", sp, "-o", op])
        if verbose:
            print("[build]", " ".join(os.path.basename(x) if x.startswith(CSRC) else x for x in cmd),
                  file=sys.stderr)
        r = subprocess.run(cmd, capture_output=True, text=True)
        err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
        if r.returncode != 0:
            raise RuntimeError("hipcc failed for %s:\n%s" % (src, err))
        if err.strip() and verbose:
            print(err, file=sys.stderr)
    cmd = [HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", LIB + ".tmp"] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    os.replace(LIB + ".tmp", LIB)
    build_io(verbose)
    for src, exe in CPP_TESTS:
        cmd = ["g++", "-std=c++17", "-O2", "-Wall", "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, src),
               "-o", os.path.join(ROOT, exe), "-L" + HERE, "-lvmc_afqmc", "-Wl,-rpath,$ORIGIN/../../vmc_amd"]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("g++ failed for %s:\n%s" % (src, r.stderr))
    return LIB


def build_io(verbose=True, sanitize=False):
    """libvmc_fcidump.so (g++, host only); returns its path, or None without HDF5.
    sanitize: the address + undefined-behaviour sanitizer build, into vmc_amd/_san/."""
    inc, lib = os.path.join(HDF5_DIR, "include"), os.path.join(HDF5_DIR, "lib")
    if not os.path.exists(os.path.join(inc, "hdf5.h")):
        if verbose:
            print("[build] no hdf5.h under %s: FCIDUMP_chol reader not built" % HDF5_DIR, file=sys.stderr)
        return None
    out = IO_LIB
    opt = ["-O2"]
    if sanitize:
        os.makedirs(os.path.join(HERE, "_san"), exist_ok=True)
        out = os.path.join(HERE, "_san", "libvmc_fcidump.so")
        # the compiler's own sanitizer runtimes, searched before the HDF5 directory (which may
        # hold other copies)
        rt = subprocess.run(["g++", "-print-file-name=libasan.so"], capture_output=True, text=True).stdout.strip()
        opt = ["-O1", "-g", "-fsanitize=address,undefined", "-fno-omit-frame-pointer", "-fno-sanitize-recover=undefined",
               "-L" + os.path.dirname(rt)]
    cmd = ["g++", "-std=c++17"] + opt + ["-Wall", "-fPIC", "-shared", "-I" + inc, "-I" + os.path.join(ROOT, "include"),
                                         IO_SRC, "-o", out + ".tmp", "-L" + lib, "-lhdf5", "-Wl,-rpath," + lib]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed for afq_fcidump.cpp:\n" + r.stderr)
    os.replace(out + ".tmp", out)
    return out


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    a = ap.parse_args()
    print(build(force=a.force))
