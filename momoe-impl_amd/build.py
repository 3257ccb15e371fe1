"""Build, in-tree, libmomoe_hip.so (gfx950) from csrc/*.hip with hipcc and the host path of the
modules, momoe_amd/_layer.so, from csrc/layer_binding.cpp against torch (host code only).

Usage: python build.py
"""
import concurrent.futures
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "momoe_amd", "libmomoe_hip.so")
LAYER = os.path.join(HERE, "momoe_amd", "_layer.so")
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # keep the compiler from emitting packed fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-value",
]


def _hipcc():
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; libmomoe_hip.so cannot be built")
    return exe


def _compile(src):
    obj = os.path.join(OBJ, os.path.basename(src).replace(".hip", ".o"))
    cmd = [_hipcc(), *FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj


def _compile_layer():
    """The object of csrc/layer_binding.cpp: host C++ against torch's headers, no device code."""
    import sysconfig
    from torch.utils import cpp_extension
    obj = os.path.join(OBJ, "layer_binding.o")
    # "cuda" adds the include directory of the ROCm that torch finds, as library_paths does below
    inc = [f"-I{p}" for p in [*cpp_extension.include_paths("cuda"), sysconfig.get_path("include")]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-Wno-deprecated-declarations",
           *inc, "-c", os.path.join(CSRC, "layer_binding.cpp"), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for layer_binding.cpp:\n{r.stderr}")
    return obj


def _link_layer(obj):
    from torch.utils import cpp_extension
    libs = cpp_extension.library_paths("cuda")
    cmd = ["g++", "-shared", obj, "-o", LAYER, f"-L{os.path.dirname(LIB)}", "-l:libmomoe_hip.so",
           "-Wl,-rpath,$ORIGIN", *[f"-L{p}" for p in libs],
           "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python", "-lamdhip64"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of the host path failed:\n{r.stderr}")


def build_library(verbose=True):
    """Compile every csrc/*.hip and the host path and link both. Always recompiles."""
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))
    with concurrent.futures.ThreadPoolExecutor(max_workers=8) as ex:
        layer = ex.submit(_compile_layer)
        objs = list(ex.map(_compile, srcs))
        layer_obj = layer.result()
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    _link_layer(layer_obj)
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources and {LAYER}")
    return LIB


if __name__ == "__main__":
    build_library()
    sys.exit(0)
