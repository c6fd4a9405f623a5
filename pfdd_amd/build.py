"""Build recipe for libpfdd_gpu.so (gfx950) and the pfdd driver, in-tree.

    python -m pfdd_amd.build            # or __graft_entry__.build()
    python -m pfdd_amd.build --incremental   # recompile only objects older than their sources

hipcc cross-compiles for gfx950 without a GPU.  Every HIP compile line carries
-Xclang -target-feature -Xclang -packed-fp32-ops (packed FP32 ops disabled).
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INC = os.path.join(ROOT, "include")
BUILD = os.path.join(ROOT, "_build")
LIB = os.path.join(PKG, "libpfdd_gpu.so")
DRIVER = os.path.join(PKG, "pfdd")
ARCH = os.environ.get("PFDD_OFFLOAD_ARCH", "gfx950")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
HIP_FLAGS = ["-O3", "-std=c++17", f"--offload-arch={ARCH}", "-fPIC", "-Wall", "-Wno-unused-function",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", f"-I{INC}", f"-I{CSRC}"]
# (source, object, extra flags): the reduced-basis kernels build as one unit per
# component count and kind, in parallel with the rest
HIP_UNITS = [("pfdd_api.hip", "pfdd_api.hip.o", [])] + [
    ("pfdd_reduced.hip", f"pfdd_reduced_{k}{r}.o", [f"-DPFDD_RED_R={r}", f"-DPFDD_RED_KIND={k}"])
    for k in range(4) for r in range(1, 7)] + [
    ("pfdd_reduced.hip", f"pfdd_reduced_{k}.o", [f"-DPFDD_RED_KIND={k}"]) for k in (4, 5, 6)]
C_SOURCES = ["pfdd_setup.c"]


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = "\n".join(l for l in (r.stdout + r.stderr).splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"build step failed: {' '.join(cmd)}\n{out}")
    return out


def _fresh(obj, src):
    """obj exists and is newer than src and the headers its dependency file names."""
    dep = obj + ".d"
    if not os.path.exists(obj) or not os.path.exists(dep):
        return False
    with open(dep) as fh:
        names = [n for n in fh.read().replace("\\\n", " ").split() if not n.endswith(":") and n.startswith(ROOT)]
    t = os.path.getmtime(obj)
    return all(os.path.exists(d) and os.path.getmtime(d) < t for d in names + [src])


def build(verbose=False, incremental=False):
    os.makedirs(BUILD, exist_ok=True)
    objs = []
    for s in C_SOURCES:
        o = os.path.join(BUILD, s + ".o")
        objs.append(o)
        if incremental and _fresh(o, os.path.join(CSRC, s)):
            continue
        _run(["gcc", "-O2", "-fPIC", "-std=c99", "-Wall", f"-I{INC}", "-MMD", "-MF", o + ".d", "-c",
              os.path.join(CSRC, s), "-o", o])

    def compile_unit(unit):
        src, obj, flags = unit
        o = os.path.join(BUILD, obj)
        if not (incremental and _fresh(o, os.path.join(CSRC, src))):
            out = _run([HIPCC] + HIP_FLAGS + flags + ["-MMD", "-MF", o + ".d", "-c", os.path.join(CSRC, src), "-o", o])
            if verbose and out.strip():
                print(out)
        return o

    with ThreadPoolExecutor(min(len(HIP_UNITS), os.cpu_count() or 1, 8)) as ex:
        objs += list(ex.map(compile_unit, HIP_UNITS))
    tmp = LIB + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC"] + objs + ["-o", tmp])
    os.replace(tmp, LIB)
    drv_src = os.path.join(PKG, "driver", "pfdd_main.c")
    if os.path.exists(drv_src):
        _run(["gcc", "-O2", "-std=c99", "-Wall", f"-I{INC}", drv_src, "-o", DRIVER, f"-L{PKG}", "-lpfdd_gpu",
              "-Wl,-rpath,$ORIGIN", "-lm"])
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv, incremental="--incremental" in sys.argv))
