"""Builds memilio_amd/libmgo.so (host engine + gfx950 kernels) with hipcc, in tree."""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libmgo.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

COMMON = ["-O3", "-std=c++20", "-fPIC", "-Wall", "-Wno-unused-function", f"--offload-arch={ARCH}",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def _stale(obj, deps):
    return not os.path.exists(obj) or any(os.path.getmtime(d) > os.path.getmtime(obj) for d in deps)


# translation units: (source, object, extra flags, further dependencies); the kernels compile as shards
UNITS = [("mgo_kernels.hip", f"mgo_kernels_{k}.o", [f"-DMGO_SHARD={k}"], []) for k in range(15)]
UNITS.append(("mgo_host.cpp", "mgo_host.o", ["-x", "hip", "-ffp-contract=off"], ["mgo_serve.inc"]))


def build(verbose=False, only_changed=False):
    """Compile the translation units (in parallel) and link libmgo.so; with only_changed, an object newer than
    its sources and headers is reused."""
    objdir = os.path.join(HERE, "_obj")
    os.makedirs(objdir, exist_ok=True)
    headers = [os.path.join(CSRC, h) for h in ("mgo_internal.h", "mgo_npi.h")]
    headers.append(os.path.join(HERE, "..", "include", "mgo.h"))
    objs, cmds = [], []
    for src, name, extra, deps in UNITS:
        obj = os.path.join(objdir, name)
        objs.append(obj)
        if only_changed and not _stale(obj, [os.path.join(CSRC, d) for d in [src, *deps]] + headers):
            continue
        cmds.append([HIPCC, *COMMON, *extra, "-c", os.path.join(CSRC, src), "-o", obj])
    # the largest shards first
    cmds.sort(key=lambda c: not any(f"MGO_SHARD={k}" in " ".join(c) for k in (9, 10, 11, 12, 14)))

    def compile_one(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)

    with ThreadPoolExecutor(max(1, min(8, os.cpu_count() or 1, int(os.environ.get("MAX_JOBS", 8))))) as pool:
        list(pool.map(compile_one, cmds))
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", OUT + ".tmp", *objs, "-lpthread"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(OUT + ".tmp", OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv, only_changed="--changed" in sys.argv))
