"""ctypes binding of ``libminit_hip.so`` (the C ABI declared in include/minit_hip.h).

The reference binds each generated launcher with ``import_symbol``, which reads
ctypes argument types from a stub's annotations (minit/compiler/cxx.py:39-59).
Here the prototypes are listed once, every function returns an ``int`` status,
and a non-zero status raises :class:`HipError` carrying ``mh_last_error()``.
There is no fallback: if the library is missing, loading raises.

``call`` is the extension module ``_binding`` (csrc/binding.cpp, built next to the
library): it converts plain numbers and pointers itself and hands every other call to
:func:`_call_general`, the ctypes path.  Without the module that path takes every call.
"""
import ctypes
import importlib.util
import os
import sys
import sysconfig
from ctypes import POINTER, c_char_p, c_double, c_float, c_int, c_size_t, c_uint32, c_uint64, c_void_p

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("MINIT_HIP_LIB") or os.path.join(_HERE, "libminit_hip.so")


class HipError(RuntimeError):
    pass


_P = c_void_p
PROTOTYPES = {
    # name: (restype, argtypes)
    "mh_abi_version": (c_int, []),
    "mh_last_error": (c_char_p, []),
    "mh_device_count": (c_int, [POINTER(c_int)]),
    "mh_device_info": (c_int, [POINTER(c_int), POINTER(c_int), POINTER(c_size_t), POINTER(c_size_t),
                               POINTER(c_int), c_char_p, c_size_t]),
    "mh_malloc": (c_int, [POINTER(c_void_p), c_size_t]),
    "mh_free": (c_int, [_P]),
    "mh_host_malloc": (c_int, [POINTER(c_void_p), c_size_t]),
    "mh_host_free": (c_int, [_P]),
    "mh_memcpy": (c_int, [_P, _P, c_size_t, _P]),
    "mh_memset": (c_int, [_P, c_int, c_size_t, _P]),
    "mh_stream_create": (c_int, [POINTER(c_void_p)]),
    "mh_stream_destroy": (c_int, [_P]),
    "mh_stream_synchronize": (c_int, [_P]),
    "mh_device_synchronize": (c_int, []),
    "mh_event_create": (c_int, [POINTER(c_void_p)]),
    "mh_event_destroy": (c_int, [_P]),
    "mh_event_record": (c_int, [_P, _P]),
    "mh_event_synchronize": (c_int, [_P]),
    "mh_event_elapsed_ms": (c_int, [POINTER(c_float), _P, _P]),
    "mh_copy_kernel": (c_int, [_P, _P, _P, c_size_t]),
    "mh_gptq_unpack": (c_int, [_P, _P, _P, c_size_t, c_size_t, c_int, c_int]),
    "mh_gptq_dequant": (c_int, [_P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int]),
    "mh_gptq_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int]),
    "mh_gptq_gemv": (c_int, [_P, _P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int, c_int, _P, c_size_t]),
    "mh_gptq_gemm": (c_int, [_P, _P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int, c_int, _P, c_size_t]),
    "mh_gptq_matmul": (c_int, [_P, _P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int, c_int, _P, c_size_t]),
    "mh_gptq_linear": (c_int, [_P, _P, _P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int, c_int, _P, c_size_t]),
    "mh_gptq_static_scratch_bytes": (c_size_t, []),
    "mh_gptq_matmul_static": (c_int, [_P, _P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int, c_int]),
    "mh_gptq_silu_pairs_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int]),
    "mh_gptq_matmul_silu_pairs": (c_int, [_P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int, c_int, _P, c_size_t]),
    "mh_f16_matmul_nk": (c_int, [_P, _P, _P, _P, c_int, c_int, c_int]),
    "mh_f16_matmul_nk_batched": (c_int, [_P, _P, _P, _P, c_int, c_int, c_int, c_int]),
    "mh_f16_matmul_tile": (c_int, [c_int, c_int, c_int, c_int]),
    "mh_i8_gemm": (c_int, [_P, _P, _P, _P, _P, _P, _P, c_int, c_int, c_int]),
    "mh_i8_gemm_tile": (c_int, [c_int, c_int, c_int]),
    "mh_i8_transpose": (c_int, [_P, _P, _P, c_int, c_int]),
    "mh_gptq_permute_rows": (c_int, [_P, _P, _P, _P, c_int, c_int, c_int]),
    "mh_rms_norm": (c_int, [_P, _P, _P, _P, c_size_t, c_size_t, c_size_t, c_double, c_int]),
    "mh_rope": (c_int, [_P, _P, _P, _P, _P, _P, c_size_t, c_size_t, c_size_t, c_size_t, c_int]),
    "mh_softmax": (c_int, [_P, _P, _P, c_size_t, c_size_t, c_size_t, c_int]),
    "mh_softmax_causal": (c_int, [_P, _P, _P, c_size_t, c_size_t, c_size_t, c_size_t, c_float, c_int]),
    "mh_sum": (c_int, [_P, _P, _P, c_size_t, c_size_t, c_size_t, c_int]),
    "mh_max": (c_int, [_P, _P, _P, c_size_t, c_size_t, c_size_t, c_int]),
    "mh_mean": (c_int, [_P, _P, _P, c_size_t, c_size_t, c_size_t, c_int]),
    "mh_sigmoid": (c_int, [_P, _P, _P, c_size_t, c_int]),
    "mh_gather_columns": (c_int, [_P, _P, _P, _P, c_size_t, c_size_t, c_int]),
    "mh_multiply": (c_int, [_P, _P, _P, _P, c_size_t, c_int]),
    "mh_add": (c_int, [_P, _P, _P, _P, c_size_t, c_int]),
    "mh_silu_mul": (c_int, [_P, _P, _P, _P, c_size_t, c_int, c_int]),
    "mh_add_bias": (c_int, [_P, _P, _P, c_size_t, c_size_t, c_int]),
    "mh_add_rms_norm": (c_int, [_P, _P, _P, _P, _P, c_int, c_int, c_float]),
    "mh_argmax": (c_int, [_P, _P, _P, c_int, c_int]),
    "mh_attn_decode_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int]),
    "mh_attn_decode": (c_int, [_P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int, c_int, _P, c_size_t]),
    "mh_rope_kv_append": (c_int, [_P, _P, _P, _P, _P, _P, _P, _P, c_int, c_int, c_int, c_int, c_int]),
    "mh_llama_create": (c_int, [POINTER(c_void_p), _P]),
    "mh_llama_destroy": (c_int, [_P]),
    "mh_llama_set_layer": (c_int, [_P, c_int, _P]),
    "mh_llama_set_globals": (c_int, [_P, _P, _P, _P, _P, _P]),
    "mh_llama_scratch_bytes": (c_size_t, [_P, c_int]),
    "mh_llama_norm_clamped": (c_int, [_P, _P, c_int, _P, POINTER(c_int)]),
    "mh_llama_decode": (c_int, [_P, _P, c_int, _P, _P, c_int, _P, _P, _P, c_size_t]),
    "mh_llama_decode_graph": (c_int, [_P, _P, c_int, _P, _P, c_int, _P, _P, _P, c_size_t]),
    "mh_synth_u32": (c_int, [_P, _P, c_size_t, c_uint64]),
    "mh_synth_subwords": (c_int, [_P, _P, c_size_t, c_int, c_uint32, c_uint32, c_uint64]),
    "mh_synth_normal": (c_int, [_P, _P, c_size_t, c_float, c_float, c_int, c_float, c_uint64, c_int]),
    "mh_synth_i8": (c_int, [_P, _P, c_size_t, c_int, c_int, c_uint64]),
}

# functions whose return value is not a status code
_NOT_STATUS = {"mh_abi_version", "mh_i8_gemm_tile", "mh_f16_matmul_tile", "mh_last_error", "mh_gptq_workspace_bytes", "mh_gptq_static_scratch_bytes", "mh_gptq_silu_pairs_workspace_bytes", "mh_llama_scratch_bytes",
               "mh_attn_decode_workspace_bytes"}

DTYPE_CODES = {"float16": 0, "bfloat16": 1, "float32": 2}

# by its full name and not as any _binding: one without the interpreter's tag may be compiled for another
_BINDING_PATH = os.path.join(_HERE, "_binding" + sysconfig.get_config_var("EXT_SUFFIX"))
_binding = None   # the extension module, once it is there
_cdll = None


def _load_binding() -> None:
    global _binding
    spec = importlib.util.spec_from_file_location(f"{__package__}._binding", _BINDING_PATH)
    try:
        module = importlib.util.module_from_spec(spec)
    except ImportError:   # not built (yet)
        return
    spec.loader.exec_module(module)
    module.set_hooks(_call_general, _failed)
    sys.modules[spec.name] = _binding = module


def _signature(restype, argtypes) -> str:
    """The codes ctypes has for the types ("P" for every pointer); the module binds what it was compiled for."""
    return "".join(t._type_ if isinstance(t._type_, str) else "P" for t in (restype, *argtypes))


def _entries(lib: ctypes.CDLL) -> dict:
    return {name: (ctypes.cast(getattr(lib, name), c_void_p).value, _signature(*types)) for name, types in PROTOTYPES.items()}


def cdll() -> ctypes.CDLL:
    """Loads the shared library (once).  Raises if it has not been built."""
    global _cdll
    if _cdll is None:
        if not os.path.exists(LIB_PATH):
            raise HipError(
                f"{LIB_PATH} is missing: build it with `python -m minit_amd.build` "
                "(there is no CPU fallback for this path)")
        lib = ctypes.CDLL(LIB_PATH)
        for name, (restype, argtypes) in PROTOTYPES.items():
            fn = getattr(lib, name)
            fn.restype = restype
            fn.argtypes = argtypes
        _cdll = lib
        if _binding is None:   # a process that has imported the package before it was built
            _load_binding()
        if _binding is not None:
            _binding.bind(_entries(lib))
    return _cdll


def last_error() -> str:
    return cdll().mh_last_error().decode(errors="replace")


_functions = {}   # name -> bound function of the loaded library


def _failed(name: str, rc: int):
    raise HipError(f"{name} failed ({rc}): {last_error()}")


def _call_general(name: str, *args):
    """Calls ``name`` and raises :class:`HipError` on a non-zero status."""
    fn = _functions.get(name)
    if fn is None:
        fn = _functions[name] = getattr(cdll(), name)
    rc = fn(*args)
    if rc and name not in _NOT_STATUS:
        _failed(name, rc)
    return rc


def _call_late(name: str, *args):
    """``call`` where the module was not there at import: other modules hold on to this function, so it looks each time."""
    return (_call_general if _binding is None else _binding.call)(name, *args)


_load_binding()
call = _call_late if _binding is None else _binding.call


def device_count() -> int:
    n = c_int(0)
    try:
        call("mh_device_count", ctypes.byref(n))
    except HipError:
        return 0
    return n.value


def device_info() -> dict:
    cus, wave, clock = c_int(0), c_int(0), c_int(0)
    mem, lds = c_size_t(0), c_size_t(0)
    name = ctypes.create_string_buffer(256)
    call("mh_device_info", ctypes.byref(cus), ctypes.byref(wave), ctypes.byref(mem), ctypes.byref(lds),
         ctypes.byref(clock), name, 256)
    return {"name": name.value.decode(), "compute_units": cus.value, "wavefront": wave.value,
            "total_mem": mem.value, "lds_per_block": lds.value, "clock_khz": clock.value}
