"""ctypes binding of libgenbmm_gfx950.so and the argument checks in front of it.

Takes the place of the reference's pybind11 module `_genbmm`
(matmul_cuda.cpp:165-172).  The reference checks `is_cuda` and `is_contiguous`
and raises RuntimeError (matmul_cuda.cpp:65-67); the checks here raise
RuntimeError for the same conditions and additionally for dtype / shape
disagreement, which the reference leaves to undefined behaviour.

There is no CPU path: calling any op without the library, or with CPU tensors,
raises.
"""
import ctypes
import importlib.util
import os
import warnings

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "lib", "libgenbmm_gfx950.so")

_c_float_p = ctypes.c_void_p
_c_int_p = ctypes.c_void_p
_i = ctypes.c_int
_u64 = ctypes.c_uint64
_vp = ctypes.c_void_p

_DENSE_DIMS = [_i, _i, _i, _i, _vp]  # B, M, K, N, stream
_BAND = [_c_float_p, _i, _i, _c_float_p, _i, _i]  # a, a_lu, a_ld, b, b_lu, b_ld

# name -> argtypes (every function returns int unless noted); mirrors
# include/genbmm_gfx950.h
SIGNATURES = {
    "genbmm_logbmm_fwd": [_c_float_p] * 4 + _DENSE_DIMS,
    "genbmm_logbmm_bwd": [_c_float_p] * 7 + _DENSE_DIMS,
    "genbmm_logbmm_fwd_static": [_c_float_p] * 3 + _DENSE_DIMS,
    "genbmm_logbmm_fwd_path": [_c_float_p] * 4 + [_i, _i, _i, _i, _i, _vp],  # ..., B, M, K, N, path, stream
    "genbmm_logbmm_bwd_path": [_c_float_p] * 7 + [_i, _i, _i, _i, _i, _vp],
    "genbmm_logbmm_bwdbwd": [_c_float_p] * 9 + _DENSE_DIMS,
    "genbmm_logbmm_bwdbwd_ws": [_c_float_p] * 10 + _DENSE_DIMS,
    "genbmm_maxbmm_fwd": [_c_float_p] * 3 + [_c_int_p] + _DENSE_DIMS,
    "genbmm_prodmaxbmm_fwd": [_c_float_p] * 3 + [_c_int_p, _c_float_p] + _DENSE_DIMS,
    "genbmm_samplebmm_fwd": [_c_float_p] * 3 + [_c_int_p, _c_float_p, _u64, _u64] + _DENSE_DIMS,
    "genbmm_argmax_bwd": [_c_int_p] + [_c_float_p] * 3 + _DENSE_DIMS,
    "genbmm_prodmax_bwd": [_c_float_p] * 2 + [_c_int_p] + [_c_float_p] * 4 + _DENSE_DIMS,
    "genbmm_banded_fwd": _BAND + [_c_float_p, _c_int_p, _c_float_p, _i, _i, _i, _vp],
    "genbmm_banded_sample_fwd": _BAND + [_c_float_p, _c_int_p, _c_float_p, _u64, _u64, _i, _i, _vp],
    "genbmm_banded_bwd": _BAND + [_c_float_p, _c_int_p] + [_c_float_p] * 4 + [_i, _i, _i, _vp],
    "genbmm_banded_bwd_scratch": _BAND + [_c_float_p, _c_int_p] + [_c_float_p] * 5 + [_i, _i, _i, _vp],
    "genbmm_banded_bwdbwd": _BAND + [_c_float_p] * 7 + [_i, _i, _vp],
    "genbmm_logbmm_fwd_f64": [_c_float_p] * 3 + _DENSE_DIMS,
    "genbmm_logbmm_bwd_f64": [_c_float_p] * 6 + _DENSE_DIMS,
    "genbmm_logbmm_bwdbwd_f64": [_c_float_p] * 9 + _DENSE_DIMS,
    "genbmm_maxbmm_fwd_f64": [_c_float_p] * 3 + [_c_int_p] + _DENSE_DIMS,
    "genbmm_prodmaxbmm_fwd_f64": [_c_float_p] * 3 + [_c_int_p] + _DENSE_DIMS,
    "genbmm_samplebmm_fwd_f64": [_c_float_p] * 3 + [_c_int_p, _u64, _u64] + _DENSE_DIMS,
    "genbmm_argmax_bwd_f64": [_c_int_p] + [_c_float_p] * 3 + _DENSE_DIMS,
    "genbmm_prodmax_bwd_f64": [_c_float_p] * 2 + [_c_int_p] + [_c_float_p] * 3 + _DENSE_DIMS,
    "genbmm_banded_fwd_f64": _BAND + [_c_float_p, _c_int_p, _i, _i, _i, _vp],
    "genbmm_banded_sample_fwd_f64": _BAND + [_c_float_p, _c_int_p, _u64, _u64, _i, _i, _vp],
    "genbmm_banded_bwd_f64": _BAND + [_c_float_p, _c_int_p] + [_c_float_p] * 3 + [_i, _i, _i, _vp],
    "genbmm_banded_bwdbwd_f64": _BAND + [_c_float_p] * 7 + [_i, _i, _vp],
    "genbmm_band_shift": [_c_float_p, _c_float_p] + [_i] * 6 + [ctypes.c_float, _vp],
    "genbmm_band_op": _BAND + [_c_float_p, _i, _i, _i, ctypes.c_float, _vp],
    "genbmm_band_transpose": [_c_float_p, _c_float_p, _i, _i, _i, _i, _vp],
    "genbmm_band_to_dense": [_c_float_p, _c_float_p, _i, _i, _i, _i, ctypes.c_float, _vp],
    "genbmm_band_from_dense": [_c_float_p, _c_float_p, _i, _i, _i, _i, _i, _vp],
}
# Entry points that also exist for float16 (`*_f16`) and bfloat16 (`*_bf16`) tensors: the same
# arguments, the caller's tensors in that type, every workspace still float32.
HALF_VARIANTS = ("genbmm_logbmm_fwd", "genbmm_logbmm_bwd", "genbmm_logbmm_fwd_path", "genbmm_logbmm_bwd_path",
                 "genbmm_maxbmm_fwd", "genbmm_prodmaxbmm_fwd", "genbmm_samplebmm_fwd", "genbmm_argmax_bwd",
                 "genbmm_prodmax_bwd", "genbmm_logbmm_bwdbwd_ws", "genbmm_banded_fwd", "genbmm_banded_sample_fwd", "genbmm_banded_bwd",
                 "genbmm_banded_bwd_scratch")
for _name in HALF_VARIANTS:
    for _suffix in ("_f16", "_bf16"):
        SIGNATURES[_name + _suffix] = SIGNATURES[_name]
for _suffix in ("_f16", "_bf16"):  # one more buffer than the float function: t_scratch (B * n * Wo floats)
    SIGNATURES["genbmm_banded_bwdbwd" + _suffix] = _BAND + [_c_float_p] * 8 + [_i, _i, _vp]
HALF_SUFFIX = {torch.float16: "_f16", torch.bfloat16: "_bf16"}
_ELEMENTS = (torch.float32, torch.float64) + tuple(HALF_SUFFIX)
STRING_FUNCS = {"genbmm_version": [], "genbmm_error_string": [_i]}
INT_FUNCS = {"genbmm_logbmm_fwd_pieces": [_i, _i, _i, _i], "genbmm_maxbmm_fwd_pieces": [_i, _i, _i, _i],
             "genbmm_banded_on_matrix_cores": [_i, _i, _i, _i, _i, _i]}
SIZE_FUNCS = {"genbmm_logbmm_stats_size": [_i, _i, _i, _i],
              "genbmm_logbmm_bwdbwd_ws_size": [_i, _i, _i, _i],
              "genbmm_logbmm_stats_size_path": [_i, _i, _i, _i, _i],
              "genbmm_samplebmm_stats_size": [_i, _i, _i, _i],
              "genbmm_logbmm_static_limit": [],
              "genbmm_banded_workspace_size": [_i, _i, _i, _i, _i, _i],
              "genbmm_banded_scratch_size": [_i, _i, _i, _i, _i, _i]}

_lib = None


def load():
    """Load the shared library (once). Raises RuntimeError if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            "genbmm_amd: %s is missing; build it with `python -m genbmm_amd.build` "
            "(there is no CPU or PyTorch fallback)" % LIB_PATH
        )
    # torch is imported above, so its HIP runtime (libamdhip64.so.7) is already
    # mapped and the library binds to that copy rather than loading a second one.
    lib = ctypes.CDLL(LIB_PATH)
    for name, argtypes in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.argtypes = argtypes
        fn.restype = ctypes.c_int
    for name, argtypes in STRING_FUNCS.items():
        fn = getattr(lib, name)
        fn.argtypes = argtypes
        fn.restype = ctypes.c_char_p
    for name, argtypes in INT_FUNCS.items():
        fn = getattr(lib, name)
        fn.argtypes = argtypes
        fn.restype = ctypes.c_int
    for name, argtypes in SIZE_FUNCS.items():
        fn = getattr(lib, name)
        fn.argtypes = argtypes
        fn.restype = ctypes.c_size_t
    _lib = lib
    host()
    return lib


_host = None    # the extension; False: it does not load


def host():
    """The extension with the eager products' autograd nodes (csrc/host.cpp), loaded once; None where none was built for
    this torch and this Python, or where it does not load.  genmul's Functions then carry every call, with the same
    results and more host time."""
    global _host
    load()      # the library it is linked to; the first call of it comes here itself
    if _host is None:
        from . import build

        spec = importlib.util.spec_from_file_location("genbmm_amd.lib._host", build.host_path())
        try:
            module = importlib.util.module_from_spec(spec)
            spec.loader.exec_module(module)
            _host = module
        except ImportError as e:
            _host = False
            warnings.warn("genbmm_amd: small products take longer than they need to, without the host extension "
                          "(%s); build it with `python -m genbmm_amd.build`" % e, RuntimeWarning, stacklevel=2)
    return _host or None


def version():
    return load().genbmm_version().decode()


def check(code, what):
    if code != 0:
        msg = load().genbmm_error_string(code).decode()
        raise RuntimeError("genbmm_amd: %s failed (%d): %s" % (what, code, msg))


def stream_of(t):
    return ctypes.c_void_p(torch.cuda.current_stream(t.device).cuda_stream)


def dense(t):
    """t as the kernels read it, by differentiable torch operations: contiguous, and written out if it carries
    torch's lazy negative bit (`z.conj().imag`), which `contiguous` keeps where the strides already fit."""
    if _host and _host.is_dense(t):
        return t
    t = t.contiguous()
    return t.resolve_neg() if t.is_neg() else t


def ptr(t):
    return ctypes.c_void_p(addr(t))


def addr(t):
    """The address of t's memory as a plain integer (None: NULL), which the declared argument types take as well as
    a pointer (`ptr`).  Refused where the memory holds the values with the other sign."""
    if t is None:
        return None
    if _host:
        return _host.address(t)
    if t.is_neg():
        raise RuntimeError("genbmm_amd: a tensor with the lazy negative bit has no memory that holds its values")
    return t.data_ptr()


def call(name, t, *args):
    """The library function `name` on t's device and that device's current stream.  The device is
    switched only where it is another one, and the stream's handle is read without a Stream object
    around it: 5.4 -> 1.5 us of host time for a call that launches nothing, two such calls in a small
    product's forward and backward."""
    fn = getattr(_lib or load(), name)
    index = t.get_device()
    if index == torch.cuda.current_device():
        code = fn(*args, torch._C._cuda_getCurrentRawStream(index))
    else:
        with torch.cuda.device(t.device):  # (refuses tensors that are on no device)
            code = fn(*args, torch._C._cuda_getCurrentRawStream(index))
    if code != 0:
        check(code, name)


def require(t, name, dtype=torch.float32, ndim=3, device=None):
    """Device / layout / dtype checks (reference CHECK_INPUT, matmul_cuda.cpp:65-67)."""
    if not isinstance(t, torch.Tensor):
        raise RuntimeError("%s must be a tensor" % name)
    if not t.is_cuda:
        raise RuntimeError("%s must be a CUDA tensor" % name)
    if not t.is_contiguous():
        raise RuntimeError("%s must be contiguous" % name)
    if t.dtype != dtype:
        raise RuntimeError("%s must be %s, got %s" % (name, dtype, t.dtype))
    if ndim is not None and t.dim() != ndim:
        raise RuntimeError("%s must have %d dimensions, got %d" % (name, ndim, t.dim()))
    if device is not None and t.device != device:
        raise RuntimeError("%s is on %s, expected %s" % (name, t.device, device))
    return t


def dense_dims(a, b):
    """(B, M, K, N) of a (B,M,K) x (B,K,N) product, with agreement checks; a's element
    type (float32, float64, float16 or bfloat16) is the one both must have."""
    if not (isinstance(a, torch.Tensor) and isinstance(b, torch.Tensor) and a.is_cuda and b.is_cuda
            and a.dtype == b.dtype and a.dtype in _ELEMENTS and a.dim() == 3 and b.dim() == 3
            and a.is_contiguous() and b.is_contiguous() and a.get_device() == b.get_device()):
        # one check after the other, for the message
        dtype = torch.float32
        if isinstance(a, torch.Tensor) and (a.dtype == torch.float64 or a.dtype in HALF_SUFFIX):
            dtype = a.dtype
        require(a, "a", dtype=dtype)
        require(b, "b", dtype=dtype, device=a.device)
    B, M, K = a.shape
    if b.shape[0] != B or b.shape[1] != K:
        raise RuntimeError(
            "shape mismatch: a is %s, b is %s" % (tuple(a.shape), tuple(b.shape))
        )
    return B, M, K, b.shape[2]
