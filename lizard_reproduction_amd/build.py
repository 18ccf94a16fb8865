"""Build liblizard_hip.so for gfx950 with hipcc, and the extension module over
it with g++ (in-tree, no JIT cache).

    python -m lizard_reproduction_amd.build

Each .hip source in csrc/ is compiled to an object in parallel, then linked
into ``lizard_reproduction_amd/_lib/liblizard_hip.so``; csrc/torch_ops.cpp, host
code against torch's headers, becomes ``_lib/lizard_torch.so``, which finds the
library beside itself.
"""
import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "_lib")
LIBNAME = "liblizard_hip.so"
MODULENAME = "lizard_torch.so"
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # keep hand-written/auto-generated packed fp32 ops out of the device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-munsafe-fp-atomics", "-Wall", "-Wno-unused-function",
]


def hipcc():
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build")
    return path


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src, obj):
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {os.path.basename(src)}:\n{proc.stderr}")
    return obj


def _compile_module(src, obj):
    """The extension module's object (host code only)."""
    import torch
    from torch.utils import cpp_extension
    includes = cpp_extension.include_paths("cuda") + [sysconfig.get_paths()["include"]]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           *(f"-isystem{path}" for path in includes), "-c", src, "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"g++ failed on {os.path.basename(src)}:\n{proc.stderr}")
    return obj


def _link_module(obj):
    from torch.utils import cpp_extension
    out = os.path.join(LIBDIR, MODULENAME)
    tmp = out + ".tmp"
    cmd = ["g++", "-shared", "-fPIC", obj, "-o", tmp,
           *(f"-L{path}" for path in cpp_extension.library_paths("cuda")), "-L" + LIBDIR,
           "-l:" + LIBNAME, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch",
           "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stderr}")
    os.replace(tmp, out)
    return out


def build(verbose=True):
    """Compile every source and link the library and the module over it;
    returns the library's path."""
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    srcs = sources()
    objs = [os.path.join(objdir, os.path.basename(s)[:-4] + ".o") for s in srcs]
    module_obj = os.path.join(objdir, "torch_ops.o")
    workers = min(len(srcs) + 1, max(1, (os.cpu_count() or 4)))
    with concurrent.futures.ThreadPoolExecutor(workers) as pool:
        module = pool.submit(_compile_module, os.path.join(CSRC, "torch_ops.cpp"), module_obj)
        list(pool.map(_compile, srcs, objs))
        module.result()
    out = os.path.join(LIBDIR, LIBNAME)
    tmp = out + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stderr}")
    os.replace(tmp, out)
    module_out = _link_module(module_obj)
    if verbose:
        print(f"built {out} and {module_out}")
    return out


if __name__ == "__main__":
    try:
        build()
    except RuntimeError as err:
        print(err, file=sys.stderr)
        sys.exit(1)
