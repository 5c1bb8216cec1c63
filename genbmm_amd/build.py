"""Build step: compile the HIP sources into libgenbmm_gfx950.so (in-tree).

    python -m genbmm_amd.build

This takes the place of the reference's setup.py (setup.py:1-27, a
torch CUDAExtension named `_genbmm`): the kernels are a plain shared library with a C ABI
(include/genbmm_gfx950.h) that genbmm_amd/_lib.py loads with ctypes; beside it a small
torch extension (csrc/host.cpp, lib/_host.*.so) holds the eager products' autograd nodes.  hipcc cross-compiles for gfx950 without
a GPU being present.
"""
import glob
import os
import shutil
import subprocess
import sys
import warnings

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIBNAME = "libgenbmm_gfx950.so"
SOURCES = ["logbmm.hip", "logbmm_bb.hip", "dense_fwd.hip", "dense_bwd.hip", "banded.hip", "band_struct.hip", "f64.hip"]
# Sources that are compiled once per element type of the caller's tensors: float (entry points
# genbmm_*), IEEE binary16 (genbmm_*_f16) and bfloat16 (genbmm_*_bf16); see csrc/common.h.
_ELEMENTS = (("", 0), ("_f16", 1), ("_bf16", 2))
PER_ELEMENT = {"logbmm.hip": _ELEMENTS, "logbmm_bb.hip": _ELEMENTS, "dense_fwd.hip": _ELEMENTS, "dense_bwd.hip": _ELEMENTS,
               "banded.hip": _ELEMENTS}

# -packed-fp32-ops is switched OFF: v_pk_{add,mul,fma}_f32 are not used by any
# kernel here, and the compiler must not form them on its own either.
HIPCC_FLAGS = [
    "-O3",
    "-std=c++17",
    "--offload-arch=gfx950",
    "-fPIC",
    # multiply-add fusion only where the source spells fmaf(): kernels whose results
    # must be bit-exact round each product before adding it
    "-ffp-contract=on",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fno-gpu-rdc",
    "-Wno-unused-command-line-argument",
]


# Per-source additions.  The banded kernels keep their 16 x 16 accumulators in ordinary vector
# registers: a tile's four values are read by vector instructions right after its last matrix
# instruction, and copies to and from the accumulation registers around every step cost
# more than the registers they free.
EXTRA_FLAGS = {"banded.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def lib_path():
    return os.path.join(LIBDIR, LIBNAME)


def host_path():
    """The eager route's autograd nodes (csrc/host.cpp): a Python extension linked to the library above, built by the
    host compiler against torch's own headers.  It uses torch's C++ interface, which is no stable one: the torch
    and the Python it was built for are in its name, so that one built for others is not found."""
    import sysconfig

    import torch

    return os.path.join(LIBDIR, "_host.torch-%s%s" % (torch.__version__, sysconfig.get_config_var("EXT_SUFFIX")))


def _host_commands(obj):
    """(compile, link) commands of the host extension."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    cxx = shutil.which("g++") or "c++"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    include = cpp_extension.include_paths() + [os.path.join(rocm, "include"), sysconfig.get_paths()["include"],
                                               os.path.join(os.path.dirname(HERE), "include")]
    compile_ = [cxx, "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
                "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI]
    compile_ += [x for path in include for x in ("-isystem", path)]
    compile_ += ["-c", os.path.join(CSRC, "host.cpp"), "-o", obj]
    link = [cxx, "-shared", obj, "-o", host_path() + ".tmp", "-L" + LIBDIR, "-l:" + LIBNAME, "-L" + torch_lib,
            "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    return compile_, link


def hipcc():
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; it is needed to build " + LIBNAME)
    return exe


def build(verbose=True):
    """Compile every source for gfx950 and link the shared library; then, with torch and a host compiler there, the host
    extension, without which the package only takes longer (a RuntimeWarning says why it was not built).
    Always recompiles."""
    os.makedirs(LIBDIR, exist_ok=True)
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    cc = hipcc()

    def start(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        return subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)

    def failure(what, proc):
        """The compiler's output if it failed, else None; waits for it."""
        out = proc.communicate()[0].decode()
        return "compiler failed on %s:\n%s" % (what, out) if proc.returncode != 0 else None

    host, host_trouble = None, None
    try:
        host_compile, host_link = _host_commands(os.path.join(objdir, "host.o"))
        host = start(host_compile)
    except (ImportError, OSError) as e:  # no torch, no compiler
        host_trouble = str(e)
    procs = []
    for src in SOURCES:
        for suffix, elem in PER_ELEMENT.get(src, (("", 0),)):
            obj = os.path.join(objdir, src.replace(".hip", suffix + ".o"))
            cmd = ([cc] + HIPCC_FLAGS + EXTRA_FLAGS.get(src, []) + ["-DGENBMM_ELEM=%d" % elem, "-c",
                   os.path.join(CSRC, src), "-o", obj])
            procs.append((src + suffix, obj, start(cmd)))
    troubles = [failure(what, proc) for what, _, proc in procs]
    if host is not None:
        host_trouble = failure("host.cpp", host)
    for trouble in troubles:
        if trouble:
            raise RuntimeError(trouble)
    tmp = lib_path() + ".tmp"
    cmd = [cc, "-shared", "-fPIC", "--offload-arch=gfx950", "-fno-gpu-rdc"] + [obj for _, obj, _ in procs] + ["-o", tmp]
    trouble = failure(LIBNAME, start(cmd))
    if trouble:
        raise RuntimeError(trouble)
    os.replace(tmp, lib_path())
    for old in glob.glob(os.path.join(glob.escape(LIBDIR), "_host.*")):
        os.remove(old)                      # an earlier build's: linked to the library that has just been replaced
    if not host_trouble:
        host_trouble = failure("the link of host.cpp", start(host_link))
    if host_trouble:
        warnings.warn("genbmm_amd: %s is built, the host extension is not: %s" % (LIBNAME, host_trouble), RuntimeWarning,
                      stacklevel=2)
    else:
        os.replace(host_path() + ".tmp", host_path())
    return lib_path()


if __name__ == "__main__":
    print(build(verbose="-q" not in sys.argv))
