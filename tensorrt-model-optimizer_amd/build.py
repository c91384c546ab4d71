"""Build libmodelopt_hip.so for gfx950 with hipcc (in-tree, next to this file).

Usage: ``python build.py [-j N] [--force] [--tuning]``.  Also importable: ``build(force=False)``.

``--tuning`` builds libmodelopt_hip_tuning.so instead, compiled with -DMO_TUNING: in that build
the per-kernel occupancy caps (unused dynamic LDS) are read from the environment at every launch
(``MO_BALLAST_<kernel>`` or ``MO_BALLAST_ALL``, in KiB), which is how the caps compiled into the
product library were chosen.  ``MODELOPT_AMD_LIB=<path>`` makes the Python layer load that file.
"""

import argparse
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libmodelopt_hip.so")
LAUNCH_SRC = os.path.join(HERE, "binding", "launch.cpp")   # compiled calls of the C ABI for the Python layer
LAUNCH_LIB = os.path.join(HERE, "modelopt_amd", "_launch.so")
LAUNCH_FOR = os.path.join(OBJ, "launch.txt")   # the interpreter and torch that LAUNCH_LIB was compiled against
PROBE_SRC = os.path.join(HERE, "probe", "l2_read_probe.hip")   # measurement aid for bench.py: its own library, outside csrc/
PROBE_LIB = os.path.join(HERE, "libmodelopt_probe.so")
HEADERS = [os.path.join(CSRC, h) for h in ("common.h", "qdq_ops.h", "awq_ops.h", "nvfp4_ops.h", "blockfp_ops.h", "mfma_ops.h")] + [
    os.path.join(HERE, "..", "include", "modelopt_hip.h")]

# -ffp-contract=off: the rounding tricks rely on separately rounded fp32 multiplies and adds.
# packed-fp32-ops is switched off on purpose (v_pk_*_f32 forms are not trusted on this target).
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-ffp-contract=off",
    "-fno-fast-math", "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp")))


def _stale(out, deps):
    if not os.path.exists(out):
        return True
    t = os.path.getmtime(out)
    return any(os.path.getmtime(d) > t for d in deps)


def _compile(src, force, obj_dir, extra):
    out = os.path.join(obj_dir, os.path.splitext(src)[0] + ".o")
    path = os.path.join(CSRC, src)
    if not force and not _stale(out, [path, *HEADERS]):
        return out
    cmd = ["hipcc", *FLAGS, *extra, "-x", "hip", "-c", path, "-o", out]
    subprocess.run(cmd, check=True)
    return out


def _interpreter():
    import torch

    return f"{sys.implementation.cache_tag} {torch.__version__} {torch.__file__}"


def _launch_is_stale():
    """Older than its sources, or compiled against another torch or Python: their layouts may differ."""
    if _stale(LAUNCH_LIB, [LAUNCH_SRC, HEADERS[-1]]) or not os.path.exists(LAUNCH_FOR):
        return True
    with open(LAUNCH_FOR) as f:
        return f.read() != _interpreter()


def _build_launch():
    """The Python extension module: host code only, against the installed torch's headers."""
    import sysconfig

    import torch

    root = os.path.dirname(os.path.abspath(torch.__file__))
    include = [os.path.join(HERE, "..", "include"), os.path.join(root, "include"),
               os.path.join(root, "include", "torch", "csrc", "api", "include"),
               os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    subprocess.run(
        ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-Wno-unused-function",
         "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_API_INCLUDE_EXTENSION_H",
         f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
         "-I", include[0], *(f for d in include[1:] for f in ("-isystem", d)), LAUNCH_SRC, "-o", LAUNCH_LIB,
         "-L", os.path.join(root, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"], check=True)
    with open(LAUNCH_FOR, "w") as f:
        f.write(_interpreter())


def build(force=False, jobs=4, tuning=False):
    obj_dir = os.path.join(OBJ, "tuning") if tuning else OBJ
    lib = LIB.replace(".so", "_tuning.so") if tuning else LIB
    extra = ["-DMO_TUNING"] if tuning else []
    os.makedirs(obj_dir, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        launch = None
        if force or _launch_is_stale():   # the Python layer needs it with either library
            launch = ex.submit(_build_launch)
        objs = list(ex.map(lambda s: _compile(s, force, obj_dir, extra), _sources()))
        if launch is not None:
            launch.result()
    if force or _stale(lib, objs):
        subprocess.run(["hipcc", "-shared", "-fPIC", "--offload-arch=gfx950", *objs, "-o", lib],
                       check=True)
    if not tuning and (force or _stale(PROBE_LIB, [PROBE_SRC])):
        subprocess.run(["hipcc", *FLAGS, "-shared", "-x", "hip", PROBE_SRC, "-o", PROBE_LIB], check=True)
    return lib


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", type=int, default=4)
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--tuning", action="store_true")
    a = ap.parse_args()
    print(build(a.force, a.j, a.tuning))
    sys.exit(0)
