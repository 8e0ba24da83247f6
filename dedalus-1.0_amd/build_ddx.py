"""Build libddx.so (hipcc, gfx950) into the package directory.

Usage: python build_ddx.py [--verbose]
"""

import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "dedalus", "libddx.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed FP32 instructions are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]

# translation units: (source, definitions); compiled side by side and linked
MIX_ROW = [("double", 0), ("double", 1), ("double", 2), ("double", 3), ("float", 2), ("float", 3)]
UNITS = [("ddx.hip", []), ("ddx_closure.hip", []), ("ddx_mixed_plan.hip", []), ("ddx_row_group.hip", []),
         ("ddx_mixed_col.hip", ["-DDDX_MIX_T=double"]), ("ddx_mixed_col.hip", ["-DDDX_MIX_T=float"])] + [
    ("ddx_mixed_row.hip", ["-DDDX_MIX_T=%s" % t, "-DDDX_MIX_ND=%d" % nd]) for t, nd in MIX_ROW]


def _compile(unit, obj, verbose):
    cmd = [HIPCC] + FLAGS + unit[1] + ["-c", os.path.join(CSRC, unit[0]), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    return res.returncode, err


def build(verbose=False):
    with tempfile.TemporaryDirectory() as tmp:
        objs = [os.path.join(tmp, "%d.o" % i) for i in range(len(UNITS))]
        with ThreadPoolExecutor(max_workers=min(8, len(UNITS))) as pool:
            done = list(pool.map(lambda u: _compile(u[0], u[1], verbose), zip(UNITS, objs)))
        for rc, err in done:
            if rc != 0 or (verbose and err.strip()):
                sys.stderr.write(err + "\n")
        if any(rc != 0 for rc, _ in done):
            raise RuntimeError("hipcc failed building libddx.so")
        lib = OUT + ".tmp"
        subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", lib], check=True)
        os.replace(lib, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose="--verbose" in sys.argv))
