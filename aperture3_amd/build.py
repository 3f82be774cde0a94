"""Build the HIP library libaperture_amd.so in-tree for gfx950.

Every .hip source under csrc/ is compiled with hipcc to an object in
_build/ and linked into aperture3_amd/libaperture_amd.so; the C++ host
mirror of the reference interface (csrc/host) is compiled into the same
library and into the example driver binary.

    python -m aperture3_amd.build      # or __graft_entry__.build()
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import re
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libaperture_amd.so")
INCLUDE = os.path.abspath(os.path.join(HERE, "..", "include"))
ARCH = os.environ.get("APT_OFFLOAD_ARCH", "gfx950")

HIP_SOURCES = [
    "kern_cart_f64.hip",
    "kern_cart_mixed.hip",
    "kern_field.hip",
    "kern_init.hip",
    "kern_sort.hip",
    "kern_tile_mixed.hip",
    "kern_tile_sort.hip",
    "kern_logsph.hip",
    "kern_rt.hip",
    "kern_ffe.hip",
    "kern_batch.hip",
    "kern_diag.hip",
    "kern_1dgr.hip",
    "kern_1dgap.hip",
    "kern_ffe_cart.hip",
    "kern_ic.hip",
    "apt_context.hip",
]
HOST_SOURCES = ["host/aperture_host.cpp"]

# -ffp-contract=off keeps every FP64 expression in the order written (the
# mixed kernels re-enable contraction locally with a pragma).  Packed FP32
# instructions are disabled for the whole device build.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
    f"-I{INCLUDE}",
    f"-I{CSRC}",
]


RESOURCE_REMARKS = ["-Rpass-analysis=kernel-resource-usage"]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"),
                 "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the HIP library cannot be built")


# Kernels compiled for a stated number of waves per SIMD.  A build of the FP64
# log-spherical push that spilled vector registers to stay within its number
# gave wrong particles, so a compiler that would spill here is refused.
NO_SPILL = ("k_logsph_push", "k_push_deposit_f64_runs", "k_push_deposit_f64_win")


def spilling_kernels(remarks: str) -> list[str]:
    """The NO_SPILL kernels that the compiler's kernel-resource-usage remarks
    report vector register spills for."""
    bad, name = [], ""
    for line in remarks.splitlines():
        m = re.search(r"remark: .*?(Function Name|VGPRs Spill): (\S+)", line)
        if not m:
            continue
        if m[1] == "Function Name":
            name = m[2]
        elif m[2] != "0" and any(k in name for k in NO_SPILL):
            bad.append(f"{name}: {m[2]} spills")
    return bad


def _run(cmd: list[str]) -> None:
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                         text=True)
    out = "\n".join(l for l in res.stdout.splitlines()
                    if "packed-fp32-ops" not in l and "not a recognized feature" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"build failed: {' '.join(cmd)}\n{out}")
    spills = spilling_kernels(res.stdout)
    if spills:
        raise RuntimeError("build refused, vector registers spilled in kernels compiled "
                           "for a stated occupancy:\n" + "\n".join(spills))


# The mixed-precision kernels use the hardware FP32 reciprocal/square root
# (<= 1 ulp) instead of the correctly rounded expansions.
FILE_FLAGS = {
    "kern_tile_mixed.hip": ["-fno-hip-fp32-correctly-rounded-divide-sqrt"],
    "kern_cart_mixed.hip": ["-fno-hip-fp32-correctly-rounded-divide-sqrt"],
    "kern_batch.hip": ["-fno-hip-fp32-correctly-rounded-divide-sqrt"],
}


def build(verbose: bool = False, jobs: int | None = None) -> str:
    hipcc = _hipcc()
    os.makedirs(BUILD, exist_ok=True)
    objs = []
    cmds = []
    for src in HIP_SOURCES + HOST_SOURCES:
        obj = os.path.join(BUILD, src.replace("/", "_") + ".o")
        objs.append(obj)
        cmds.append([hipcc, *HIPCC_FLAGS, *FILE_FLAGS.get(src, []),
                     *(RESOURCE_REMARKS if src.endswith(".hip") else []), "-c",
                     os.path.join(CSRC, src), "-o", obj])
    jobs = jobs or min(8, os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        for cmd, _ in zip(cmds, ex.map(_run, cmds)):
            if verbose:
                print(" ".join(cmd))
    tmp = LIB + ".tmp"
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    # example driver built on the C++ host mirror
    drv = os.path.join(HERE, "pic_step_driver")
    _run([hipcc, "-O2", "-std=c++17", f"-I{INCLUDE}", f"-I{CSRC}",
          os.path.join(CSRC, "host", "pic_step_driver.cpp"), "-o", drv + ".tmp",
          f"-L{HERE}", "-laperture_amd", f"-Wl,-rpath,{HERE}", "-Wl,-rpath,$ORIGIN"])
    os.replace(drv + ".tmp", drv)
    ic = os.path.join(HERE, "ic_driver")
    _run([hipcc, "-O2", "-std=c++17", f"-I{INCLUDE}", f"-I{CSRC}",
          os.path.join(CSRC, "host", "ic_driver.cpp"), "-o", ic + ".tmp",
          f"-L{HERE}", "-laperture_amd", f"-Wl,-rpath,{HERE}", "-Wl,-rpath,$ORIGIN"])
    os.replace(ic + ".tmp", ic)
    build_io()
    return LIB


# HDF5 output and snapshots link the HDF5 C library; the library is built
# where the HDF5 headers are found and skipped (with a message) elsewhere.
HDF5_ROOTS = [os.environ.get("APT_HDF5_ROOT"), "/opt/conda", "/usr"]
IO_LIB = os.path.join(HERE, "libaperture_io.so")


def hdf5_root() -> str | None:
    for root in HDF5_ROOTS:
        if root and os.path.exists(os.path.join(root, "include", "hdf5.h")):
            return root
    return None


def build_io() -> str | None:
    root = hdf5_root()
    if root is None:
        print("aperture3_amd: hdf5.h not found, libaperture_io.so not built",
              file=sys.stderr)
        return None
    libdir = os.path.join(root, "lib")
    tmp = IO_LIB + ".tmp"
    # libstdc++ is linked statically: the HDF5 directory may hold an older
    # libstdc++.so that the run path would otherwise hand to the HIP runtime
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
          "-static-libstdc++", "-static-libgcc",
          f"-I{INCLUDE}", f"-I{os.path.join(root, 'include')}",
          os.path.join(CSRC, "io", "apt_io.cpp"), "-o", tmp,
          f"-L{HERE}", "-laperture_amd", f"-L{libdir}", "-lhdf5",
          "-Wl,-rpath,$ORIGIN", f"-Wl,-rpath,{libdir}"])
    os.replace(tmp, IO_LIB)
    # lab-style driver on the C++ host mirror and data_exporter.hpp
    drv = os.path.join(HERE, "pulsar_driver")
    _run(["g++", "-O2", "-std=c++17", f"-I{INCLUDE}", f"-I{os.path.join(CSRC, 'host')}",
          os.path.join(CSRC, "host", "pulsar_driver.cpp"), "-o", drv + ".tmp",
          f"-L{HERE}", "-laperture_io", "-laperture_amd", "-Wl,-rpath,$ORIGIN"])
    os.replace(drv + ".tmp", drv)
    return IO_LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
