"""ctypes binding of libhaste_hip.so, the C-ABI library declared in include/haste_hip.h.

The library must have been built (python -m haste_amd.build); there is no fallback:
loading fails loudly when it is missing.
"""
import ctypes
import functools
import os
import re

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libhaste_hip.so")
HEADER_PATH = os.path.join(os.path.dirname(_HERE), "include", "haste_hip.h")

_lib = None


class HasteHipError(RuntimeError):
    def __init__(self, code, where):
        lib = load()
        text = lib.haste_hip_error_string(code).decode()
        detail = lib.haste_hip_last_runtime_error().decode()
        super().__init__("%s failed: %s%s" % (where, text, (" [" + detail + "]") if detail else ""))
        self.code = code


def declared_symbols():
    """Names of every function include/haste_hip.h declares."""
    with open(HEADER_PATH) as f:
        text = f.read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(haste_hip_[a-z0-9_]+)\s*\(", text)))


def load():
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise ImportError(
            "libhaste_hip.so is not built: run `python -m haste_amd.build` (needs hipcc). "
            "There is no CPU fallback.")
    lib = ctypes.CDLL(LIB_PATH)
    lib.haste_hip_error_string.restype = ctypes.c_char_p
    lib.haste_hip_error_string.argtypes = [ctypes.c_int]
    lib.haste_hip_last_runtime_error.restype = ctypes.c_char_p
    lib.haste_hip_last_runtime_error.argtypes = []
    lib.haste_hip_version.restype = ctypes.c_int
    _lib = lib
    return lib


_TYPES = {"int": ctypes.c_int, "float": ctypes.c_float, "size_t": ctypes.c_size_t}
_entries = {}


def entry(name):
    """Entry point `name` with the argument types its declaration in include/haste_hip.h has: the
    arguments of a call are then converted by ctypes itself (a wrapper object per argument, made in
    Python, costs more than the rest of a short call; a package without the header does that).  None
    when the library has no such entry."""
    fn = _entries.get(name)
    if fn is None:
        try:
            fn = load()[name]  # a function object of this module's own: its argument types are nobody else's
        except AttributeError:
            return None
        fn.restype = ctypes.c_int
        parameters = _parameters().get(name)
        if parameters is not None:
            fn.argtypes = [ctypes.c_void_p if "*" in p else _TYPES[p.split()[-2]] for p in parameters]
        _entries[name] = fn
    return fn


@functools.lru_cache(maxsize=None)
def _parameters():
    if not os.path.exists(HEADER_PATH):
        return {}
    with open(HEADER_PATH) as f:
        text = re.sub(r"/\*.*?\*/", "", f.read(), flags=re.S)
    found = re.findall(r"\b(haste_hip_[a-z0-9_]+)\s*\(([^()]*)\)", text)
    return {name: [p.strip() for p in params.split(",")] for name, params in found}


def _wrapped(a):
    """An argument of an entry point whose declaration is not at hand.  Whole numbers go as 64 bits: the
    callee reads as many of them as its parameter has, and addresses need all."""
    if a is None or isinstance(a, float):
        return ctypes.c_void_p(a) if a is None else ctypes.c_float(a)
    return ctypes.c_longlong(a)


def _current_stream():
    """The address of torch's current stream: what torch.cuda.current_stream().cuda_stream is, without an object for it
    (2.5 us of a call's 13)."""
    if _raw_stream is None or not torch.cuda.is_initialized():
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(torch.cuda.current_device())


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def invoke(name, fn, values, stream=None):
    """Calls the entry point `fn` (of that name) with ints, floats and addresses, plus the stream."""
    values.append(_current_stream() if stream is None else stream)
    rc = fn(*values) if fn.argtypes is not None else fn(*map(_wrapped, values))
    if rc != 0:
        raise HasteHipError(rc, name)


def call(name, *args, stream=None):
    """Calls entry point `name` with ints/floats/tensors/addresses (None = NULL) plus the stream."""
    fn = entry(name)
    if fn is None:
        raise AttributeError("libhaste_hip.so has no entry point " + name)
    invoke(name, fn, [a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args], stream)
