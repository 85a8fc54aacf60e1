"""Build the gfx950 shared library ``bgy3d_amd/librism3d.so`` in-tree.

    python -m bgy3d_amd.build

hipcc compiles the HIP translation units for gfx950 only (cross-compiles
without a GPU); the host C++ of the 1D chi producer is built by hipcc as
plain C++.  Packed-FP32 instruction selection is disabled for device code.
"""
import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "librism3d.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

HIP_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


# (object, source, flags): the residual chain's kernels are templates with
# many instantiations, split by pass and working type to build in parallel.
UNITS = [("solver", "solver.hip", HIP_FLAGS), ("rism1d", "rism1d.cpp", None)] + [
    (f"{src}_{t[0]}", f"{src}.hip", HIP_FLAGS + [f"-DRISM_T={t}"])
    for src, types in (("chain_rows", ("double", "float")), ("chain_zpass", ("double", "float")),
                       ("chain_planes", ("double", "float")))
    for t in types]


def build(verbose=False):
    def compile_unit(unit):
        name, src, flags = unit
        out = os.path.join(CSRC, name + ".o")
        if flags is None:
            cmd = [HIPCC, "-x", "c++", "-O3", "-std=c++17", "-fPIC", "-Wall"]
        else:
            cmd = [HIPCC] + flags
        cmd += ["-c", os.path.join(CSRC, src), "-o", out]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)
        return out

    with concurrent.futures.ThreadPoolExecutor(max_workers=8) as pool:
        objs = list(pool.map(compile_unit, UNITS))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB + ".tmp"] + objs
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(LIB + ".tmp", LIB)
    for o in objs:
        os.remove(o)
    return LIB


if __name__ == "__main__":
    build(verbose="-v" in sys.argv)
    print(LIB)
