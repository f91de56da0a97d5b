"""ctypes binding of libmvme_paged.so (the C ABI declared in include/mvme_paged.h).

Plays the role of the reference's ``load_cuda_extension``
(mini_engine/kernels/cuda_extension.py:14-66): one cached handle per
process.  There is no fallback: a missing or unloadable library raises.  (The
native call path beside it is only a faster way into the same library.)
"""

from __future__ import annotations

import ctypes
import functools
import importlib.machinery
import importlib.util
import warnings

import torch

from .. import build as _build

FP16, BF16, FP32 = 0, 1, 2
OK, EINVAL, ELAUNCH, EWORKSPACE = 0, 1, 2, 3
ABI_VERSION = 2

_i64, _vp, _int, _size = ctypes.c_int64, ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t

# name -> (restype, argtypes); mirrors include/mvme_paged.h.
SIGNATURES = {
    "mvme_abi_version": (_int, []),
    "mvme_last_error": (ctypes.c_char_p, []),
    "mvme_write_kv_cache_slots": (_int, [_vp, _vp, _i64, _i64, _i64, _i64, _vp, _vp, _vp, _i64,
                                         _i64, _i64, _int, _vp]),
    "mvme_write_kv_cache_batch": (_int, [_vp, _vp, _i64, _i64, _i64, _i64, _vp, _i64, _vp, _vp, _vp,
                                         _i64, _int, _vp]),
    "mvme_write_kv_cache": (_int, [_vp, _vp, _i64, _i64, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _i64,
                                   _int, _vp]),
    "mvme_gather_kv_cache": (_int, [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp, _i64, _i64, _int,
                                    _vp]),
    "mvme_paged_attention_workspace_size": (_size, [_i64, _i64, _i64, _i64, _i64, _i64, _i64]),
    "mvme_paged_attention": (_int, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _i64,
                                    _i64, _i64, _int, _vp, _size, _vp]),
    "mvme_paged_attention_noalloc": (_int, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64,
                                            _i64, _i64, _i64, _int, _vp]),
    "mvme_paged_attention_decode_write": (_int, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64,
                                                 _i64, _i64, _i64, _int, _vp, _vp, _i64, _i64, _vp, _vp, _vp,
                                                 _vp, ctypes.c_float, _i64, _vp, _vp, _size, _vp]),
    "mvme_paged_prefill_workspace_size": (_size, [_i64] * 8 + [_int]),
    "mvme_paged_prefill_attention": (_int, [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64,
                                            _i64, _i64, _i64, _i64, _i64, _i64, _int, _vp, _size, _vp]),
    "mvme_prefill_attention_workspace_size": (_size, [_i64] * 6 + [_int]),
    "mvme_prefill_attention": (_int, [_vp, _vp, _vp, _vp] + [_i64] * 16 + [_int, _vp, _size, _vp]),
    "mvme_qk_norm_rope_write_kv": (_int, [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp, _vp, _i64, _vp,
                                          _vp, _vp, _vp, _i64, _i64, _i64, _vp, _vp, _vp, _vp, _i64, _i64,
                                          ctypes.c_float, _int, _vp]),
    "mvme_greedy_argmax_workspace_size": (_size, [_i64, _i64]),
    "mvme_greedy_argmax": (_int, [_vp, _vp, _i64, _i64, _i64, _int, _vp, _size, _vp]),
    "mvme_linear_rows": (_int, [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _int, _vp]),
}


class HipLibrary:
    """Typed handle on the shared object; every call checks its status."""

    def __init__(self, lib: ctypes.CDLL, path):
        self._lib = lib
        self.path = path
        for name, (restype, argtypes) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = restype
            fn.argtypes = argtypes
        version = lib.mvme_abi_version()
        if version != ABI_VERSION:
            raise RuntimeError(f"libmvme_paged ABI version {version}, expected {ABI_VERSION}")

    def last_error(self) -> str:
        message = self._lib.mvme_last_error()
        return message.decode() if message else ""

    def call(self, name: str, *args):
        status = getattr(self._lib, name)(*args)
        if status != OK:
            raise RuntimeError(f"{name}: {self.last_error()} (status {status})")

    def workspace_size(self, *args) -> int:
        return int(self._lib.mvme_paged_attention_workspace_size(*args))

    def prefill_workspace_size(self, *args) -> int:
        return int(self._lib.mvme_paged_prefill_workspace_size(*args))

    def dense_prefill_workspace_size(self, *args) -> int:
        return int(self._lib.mvme_prefill_attention_workspace_size(*args))

    def argmax_workspace_size(self, *args) -> int:
        return int(self._lib.mvme_greedy_argmax_workspace_size(*args))


def check_build_digest(digest_file, expected: str) -> None:
    """Refuse a library built from other sources than the ones beside it.

    ``build_library`` writes the sha256 of the HIP sources and headers next to
    the library; a missing or different digest means the library is stale.
    """
    try:
        recorded = digest_file.read_text().strip()
    except OSError as error:
        raise RuntimeError(f"no build digest at {digest_file}: rebuild the HIP library "
                           f"(python -m mini_engine_hip.build)") from error
    if recorded != expected:
        raise RuntimeError(f"stale HIP library: the sources changed since it was built "
                           f"(digest {recorded[:12]} != {expected[:12]}); rebuild with "
                           f"python -m mini_engine_hip.build")


class NoNativeCalls:
    """Stands for the native call path where it is not loaded: declines every call."""

    def _decline(self, *args):
        return None

    decode = decode_write = prefill = dense = linear = rope_slots = write_slots = _decline


# What the entry points ask first; `load_hip_extension` puts the native call
# path here.  The first call of a process therefore runs the Python code, and a
# call that is refused, or that needs no library, never loads one.
native = NoNativeCalls()


@functools.lru_cache(maxsize=1)
def load_hip_extension() -> HipLibrary:
    """Load the prebuilt library; build it first only if no build exists.

    An existing library must carry the digest of the current sources.
    """
    global native
    path = _build.library_path()
    if not path.exists():
        try:
            _build.build_library()
        except RuntimeError:
            if not path.exists():  # else only the native call path is missing
                raise
    check_build_digest(_build.digest_path(), _build.source_digest())
    try:
        lib = ctypes.CDLL(str(path))
    except OSError as error:
        raise RuntimeError(f"cannot load the HIP paged-attention library {path}: {error}") from error
    library = HipLibrary(lib, path)
    native = _bind_native(library)
    return library


# Entry points of the native call path (csrc/host_calls.cpp), in its order.
_HOST_ENTRY_POINTS = ("mvme_last_error", "mvme_paged_attention_workspace_size", "mvme_paged_attention",
                      "mvme_paged_attention_decode_write", "mvme_paged_prefill_workspace_size",
                      "mvme_paged_prefill_attention", "mvme_prefill_attention_workspace_size",
                      "mvme_prefill_attention", "mvme_write_kv_cache_slots", "mvme_linear_rows",
                      "mvme_qk_norm_rope_write_kv")


@functools.lru_cache(maxsize=1)
def _host_module():
    path = _build.host_path()
    try:
        recorded = _build.host_digest_path().read_text().strip()
    except OSError as error:
        raise RuntimeError(f"no build digest of the native call path: {error}") from error
    if recorded != _build.host_digest():
        raise RuntimeError("the native call path was built from other sources or for another torch or Python")
    loader = importlib.machinery.ExtensionFileLoader("mvme_host", str(path))
    spec = importlib.util.spec_from_file_location("mvme_host", str(path), loader=loader)
    try:
        module = importlib.util.module_from_spec(spec)
        loader.exec_module(module)
    except (ImportError, OSError) as error:
        raise RuntimeError(f"cannot load the native call path {path}: {error}") from error
    return module


def _bind_native(library):
    """The native call path on ``library``, or what declines every call: the
    Python code serves them all, so a host module that cannot be loaded costs
    time, not calls."""
    try:
        module = _host_module()
    except RuntimeError as error:
        warnings.warn(f"{error}; calls take the Python path (rebuild with python -m mini_engine_hip.build)",
                      RuntimeWarning, stacklevel=3)
        return NoNativeCalls()
    module.bind(torch._C._cuda_getCurrentRawStream,
                tuple(ctypes.cast(getattr(library._lib, name), _vp).value for name in _HOST_ENTRY_POINTS))
    return module


def native_calls():
    """The entry points' native call path: functions that run a plain call
    (dense CUDA tensors of the current device, no caller-supplied buffers, no
    host-synchronising validation) and return None for any other, which the
    Python code then checks and runs.  Measured, us per call: a decode call of
    one 128-token sequence 14.6 -> 4.6, a decode step of 8 sequences 29.0 ->
    9.8, which is then the GPU's time."""
    load_hip_extension()
    return native


def dtype_code(dtype: torch.dtype) -> int:
    if dtype == torch.float16:
        return FP16
    if dtype == torch.bfloat16:
        return BF16
    raise ValueError("HIP kernels support FP16/BF16")


def current_stream(device: torch.device) -> int:
    """Raw hipStream_t of torch's current stream on ``device``."""
    return torch.cuda.current_stream(device).cuda_stream


def ptr(tensor: torch.Tensor) -> int:
    return tensor.data_ptr()
