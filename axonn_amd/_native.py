"""ctypes binding of libaxn_gfx950.so (the C ABI declared in include/axn.h).

The library holds every kernel of the hot path; this module only marshals
pointers, sizes and the current HIP stream.  There is no fallback: when the
library is missing, loading raises, and every compute entry point needs a GPU.
"""

import ctypes
import importlib.machinery
import importlib.util
import os
import sys
import threading
import warnings

_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib", "libaxn_gfx950.so")

AXN_OK = 0
AXN_EINVAL = -1
AXN_EALIGN = -2
AXN_ESHAPE = -3
AXN_EHIP = -4
AXN_ELIMIT = -5

BF16, F16, F32 = 0, 1, 2
EPI_NONE, EPI_BIAS, EPI_BIAS_GELU, EPI_GELU = 0, 1, 2, 3
BIAS_16BIT = 0x100   # with an epilogue: the bias has the operands' 16-bit type
DY_F32, DBIAS_16BIT = 0x100, 0x200   # with the dtype of axn_dgelu_dbias: dY is fp32; dbias is not
ROUNDED = 0x100      # with F32 as an input gradient's output type: 16-bit values
ANY_SIZES = 0x100    # with the dtype of axn_gemm_swiglu_fwd: sizes that are not made of whole tiles

ABI_VERSION = 16   # another one with every change of the entry points below or of the constants above

# Every symbol include/axn.h declares: name -> (restype, argtypes)
_c = ctypes
_vp, _i64, _int, _f32, _sz = _c.c_void_p, _c.c_int64, _c.c_int, _c.c_float, _c.c_size_t
_pp, _pi64 = _c.POINTER(_c.c_void_p), _c.POINTER(_c.c_int64)


class AdamHParams(ctypes.Structure):
    """Mirror of axn_adam_hparams."""

    _fields_ = [
        ("lr_over_bc1", _f32),
        ("inv_sqrt_bc2", _f32),
        ("beta1", _f32),
        ("one_minus_beta1", _f32),
        ("beta2", _f32),
        ("one_minus_beta2", _f32),
        ("eps", _f32),
        ("weight_decay", _f32),
    ]


SCAN_RESULT_BYTES = 32  # sizeof(axn_scan_result)

SYMBOLS = {
    "axn_abi_version": (_int, []),
    "axn_last_error": (_c.c_char_p, []),
    "axn_gemm_fwd": (_int, [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _int, _vp]),
    "axn_gemm_dgrad": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _vp]),
    "axn_gemm_wgrad": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int, _vp]),
    "axn_gemm_fwd_f16": (_int, [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _int,
                                _vp]),
    "axn_gemm_bwd": (_int, [_vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64,
                            _int, _int, _vp]),
    "axn_gemm_fwd_f32out": (_int, [_vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64,
                                   _int, _vp]),
    "axn_gemm_dgrad_f16": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _vp]),
    "axn_gemm_wgrad_f16": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64, _int, _int,
                                  _vp]),
    "axn_gemm_workspace_bytes": (_sz, [_int, _i64, _i64, _i64]),
    "axn_gemm_fwd_ws": (_int, [_vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _int,
                               _vp, _sz, _vp]),
    "axn_gemm_dgrad_ws": (_int, [_vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _vp, _sz,
                                 _vp]),
    "axn_gemm_wgrad_ws": (_int, [_vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _int,
                                 _int, _vp, _sz, _vp]),
    "axn_dgelu_dbias": (_int, [_vp, _vp, _vp, _int, _vp, _i64, _i64, _i64, _int, _vp, _sz, _vp]),
    "axn_gemm_swiglu_fwd": (_int, [_vp, _vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _vp]),
    "axn_gemm_swiglu_fwd_few": (_int, [_vp, _vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _vp]),
    "axn_gemm_dgrad_pair": (_int, [_vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _vp]),
    "axn_dgelu_dbias_workspace_bytes": (_sz, [_i64, _i64]),
    "axn_swiglu_fwd": (_int, [_vp, _vp, _vp, _int, _i64, _i64, _i64, _vp]),
    "axn_swiglu_bwd": (_int, [_vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _vp]),
    "axn_embedding_fwd": (_int, [_vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _vp, _vp]),
    "axn_embedding_workspace_bytes": (_sz, [_i64, _i64]),
    "axn_embedding_bwd": (_int, [_vp, _vp, _vp, _int, _int, _i64, _i64, _i64, _i64, _i64, _i64,
                                 _int, _int, _vp, _sz, _vp]),
    "axn_embedding_renorm": (_int, [_vp, _vp, _int, _i64, _i64, _i64, _i64, _f32, _f32, _vp, _sz,
                                    _vp]),
    "axn_gemm_fwd_f32": (_int, [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _int, _vp]),
    "axn_gemm_dgrad_f32": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _vp]),
    "axn_gemm_wgrad_f32": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _int, _vp]),
    "axn_gemm_any_n": (_int, [_int, _vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _int,
                              _int, _int, _vp, _sz, _vp]),
    "axn_gemm_bwd_workspace_bytes": (_sz, [_i64, _i64, _i64, _int]),
    "axn_gemm_bwd_ws": (_int, [_vp, _vp, _vp, _vp, _vp, _int, _i64, _i64, _i64, _i64, _i64, _i64, _i64, _i64,
                               _int, _int, _vp, _sz, _vp]),
    "axn_pad_rows16": (_int, [_vp, _vp, _i64, _i64, _i64, _vp]),
    "axn_pad_rows16_to": (_int, [_vp, _vp, _i64, _i64, _i64, _i64, _vp]),
    "axn_gemm_f32_workspace_bytes": (_sz, [_int, _i64, _i64, _i64]),
    "axn_gemm_fwd_f32_ws": (_int, [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _int, _vp, _sz, _vp]),
    "axn_gemm_dgrad_f32_ws": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _vp, _sz, _vp]),
    "axn_gemm_wgrad_f32_ws": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _int, _vp, _sz, _vp]),
    "axn_mt_scan_workspace_bytes": (_sz, [_i64, _i64]),
    "axn_mt_scan": (_int, [_pp, _pi64, _i64, _int, _f32, _f32, _int, _vp, _vp, _sz, _vp]),
    "axn_mt_scan_norm": (_int, [_pp, _pi64, _i64, _int, _f32, _f32, _f32, _int, _vp, _vp, _sz, _vp]),
    "axn_mt_scan_noalloc": (_int, [_pp, _pi64, _i64, _int, _f32, _f32, _int, _vp, _vp]),
    "axn_mt_adam": (_int, [_pp, _pp, _pp, _pp, _pp, _pi64, _i64, _int, _int, _f32, _vp,
                           _c.POINTER(AdamHParams), _vp]),
    "axn_mt_scale": (_int, [_pp, _pi64, _i64, _int, _f32, _vp, _int, _vp]),
}

_lib = None
_probe_lib = None
# axn_fast.so (csrc/fast.cpp): the host side of the usual Linear calls, same kernels.  None before `load` and where it is
# not built or does not fit: every caller then goes the general way, which it also goes where a function of `fast` answers
# None.
fast = None
_lock = threading.Lock()


class AxnError(RuntimeError):
    """A call into libaxn_gfx950.so returned a non-zero status."""

    def __init__(self, code, message):
        super().__init__("libaxn_gfx950 error %d: %s" % (code, message))
        self.code = code


def lib_path():
    return _LIB_PATH


def _load_fast(lib):
    """axn_fast.so, or None.  Unlike the library it is tied to one PyTorch and one Python: built for others, or for another
    version of this package, it is left alone with a warning."""
    path = os.path.join(os.path.dirname(_LIB_PATH), "axn_fast.so")
    if not os.path.exists(path):
        return None
    try:
        import torch
    except ImportError:
        return None   # (nobody calls it)
    try:
        loader = importlib.machinery.ExtensionFileLoader("axn_fast", path)
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("axn_fast", loader))
        loader.exec_module(module)
        built, wanted = (module.ABI_VERSION, module.BUILT_FOR), (ABI_VERSION, fast_built_for(torch))
        if built != wanted:
            raise ImportError("it was built for %s, this is %s" % (built, wanted))
        module.bind(dict({name: ctypes.cast(getattr(lib, name), _vp).value for name in module.entry_points()}, check=check))
    except (ImportError, AttributeError) as error:
        warnings.warn("axn_fast.so is not used, Linear calls take more host time (%s); run "
                      "`python -m axonn_amd.csrc.build`" % error, stacklevel=3)
        return None
    dtype_code(torch.float32)   # (fills the table that callers of `fast` look types up in)
    return module


def fast_built_for(torch):
    """What axn_fast.so is built for beside the library's version."""
    return "%s, PyTorch %s" % (sys.implementation.cache_tag, torch.__version__)


def load():
    """Loads the library once and types its entry points.  Raises if it is absent."""
    global _lib, fast
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(_LIB_PATH):
            raise ImportError(
                "libaxn_gfx950.so is not built (expected at %s); run "
                "`python -m axonn_amd.csrc.build`" % _LIB_PATH
            )
        try:
            # PyTorch ships its own HIP runtime with the same soname; importing it
            # first makes this library bind to the runtime that owns torch's
            # streams and allocations.
            import torch  # noqa: F401
        except ImportError:
            pass
        lib = ctypes.CDLL(_LIB_PATH)
        if lib.axn_abi_version() != ABI_VERSION:   # (before the entry points, of which another version may lack some)
            raise ImportError(
                "libaxn_gfx950.so has ABI version %d, this package needs %d"
                % (lib.axn_abi_version(), ABI_VERSION)
            )
        for name, (restype, argtypes) in SYMBOLS.items():
            fn = getattr(lib, name)
            fn.restype = restype
            fn.argtypes = argtypes
        fast = _load_fast(lib)
        _lib = lib
    return _lib


def load_probe():
    """The benchmark-only library of streaming yardsticks (include/axn_probe.h)."""
    global _probe_lib
    if _probe_lib is None:
        path = os.path.join(os.path.dirname(_LIB_PATH), "libaxn_probe_gfx950.so")
        if not os.path.exists(path):
            raise ImportError("libaxn_probe_gfx950.so is not built (expected at %s); run "
                              "`python -m axonn_amd.csrc.build`" % path)
        load()  # binds the HIP runtime torch uses first
        lib = ctypes.CDLL(path)
        lib.axn_probe_stream.restype = _int
        lib.axn_probe_stream.argtypes = [_int, _vp, _vp, _sz, _vp]
        _probe_lib = lib
    return _probe_lib


def check(rc):
    if rc != AXN_OK:
        msg = load().axn_last_error()
        raise AxnError(rc, msg.decode("utf-8", "replace") if msg else "")


def call(name, *args):
    """Calls an int-returning entry point and raises AxnError on failure."""
    rc = getattr(_lib or load(), name)(*args)
    if rc != AXN_OK:
        check(rc)


_DTYPE_CODES = {}


def dtype_code(torch_dtype):
    if not _DTYPE_CODES:
        import torch

        _DTYPE_CODES.update({torch.bfloat16: BF16, torch.float16: F16, torch.float32: F32})
    code = _DTYPE_CODES.get(torch_dtype)
    if code is None:
        raise TypeError("unsupported dtype %s (bf16, fp16 or fp32 expected)" % torch_dtype)
    return code


def current_stream():
    """torch's current stream on the current device, a `hipStream_t` as a plain number."""
    import torch

    raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)
    if raw is not None:  # the handle itself, without building a Stream object (5-10 us less per call)
        return raw(torch.cuda.current_device())
    return torch.cuda.current_stream().cuda_stream


def ptr(t):
    """Device pointer of a tensor (None -> NULL), a plain number: the entry points' argument types convert it
    (a c_void_p object an argument made a call of 19 arguments 5.1 us, so 4.0, its launch included)."""
    return None if t is None else t.data_ptr()


def ptr_array(tensors):
    arr = (ctypes.c_void_p * max(len(tensors), 1))()
    for i, t in enumerate(tensors):
        arr[i] = t.data_ptr()
    return arr


def size_array(tensors):
    arr = (ctypes.c_int64 * max(len(tensors), 1))()
    for i, t in enumerate(tensors):
        arr[i] = t.numel()
    return arr
