"""Build librkstiff_amd.so for gfx950 with hipcc (in-tree, no JIT cache).

Translation units (rkstiff_amd/csrc): one per precision x nonlinearity x method for
the persistent stepping kernels, the host/C-ABI unit and the tableau unit.  They
compile in parallel and link into rkstiff_amd/librkstiff_amd.so.
"""
import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "librkstiff_amd.so")
BUILD = os.path.join(HERE, "_build")
ARCH = os.environ.get("RKS_OFFLOAD_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["-O3", "-std=c++17", f"--offload-arch={ARCH}", "-fPIC",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-I" + os.path.join(HERE, "..", "include"), "-Wno-unused-result"]
# (source, object name, defines): the stepping kernels once per precision x nonlinearity x method
PRECISIONS = {"f64": ("double", "double"), "mix": ("double", "float"), "f32": ("float", "float")}
METHODS = {"any": "RKS_METH_ANY", "etd35": "RKS_M_ETD35", "if34": "RKS_M_IF34"}
UNITS = [("rks_k.hip", f"rks_k_{p}_{nl}_{m}",
          [f"-DRKS_R={r}", f"-DRKS_RN={rn}", f"-DRKS_NLK=NLK_{nl.upper()}", f"-DRKS_METH={meth}",
           f"-DRKS_TABLE=rks_k_{p}_{nl}_{m}"])
         for nl in ("cubic", "advect", "hankel") for m, meth in METHODS.items() for p, (r, rn) in PRECISIONS.items()
         if not (nl == "hankel" and m == "if34")]
UNITS += [(u, u, []) for u in ("rks_2d.hip", "rks_mlp.hip", "rks_hankel.hip", "rks_dense.hip", "rks_host.hip",
                               "rks_tableau.cpp")]


def _compile(unit, verbose):
    source, name, defines = unit
    obj = os.path.join(BUILD, name + ".o")
    lang = ["-x", "hip"] if source.endswith(".hip") else []
    cmd = [HIPCC] + FLAGS + defines + lang + ["-c", os.path.join(SRC, source), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = "\n".join(line for line in (r.stdout + r.stderr).splitlines()
                     if "unknown target feature" not in line and "packed-fp32-ops" not in line)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {name}:\n{out}")
    if verbose and out.strip():
        print(out)
    return obj


def build(verbose=False, jobs=None):
    """Compile every unit (always) and link the shared library; returns its path."""
    os.makedirs(BUILD, exist_ok=True)
    jobs = jobs or min(len(UNITS), max(1, os.cpu_count() or 1))
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(lambda u: _compile(u, verbose), UNITS))
    tmp = OUT + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    t = build(verbose="-v" in sys.argv)
    print(t)
