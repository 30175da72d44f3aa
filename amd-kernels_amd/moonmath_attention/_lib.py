"""ctypes binding of ``libmoonmath_gfx950.so`` (the C ABI in include/moonmath_gfx950.h).

Replaces the reference's pybind ``moonmath_attention._C`` extension
(moonmath reference csrc/attention_api.cpp:441-473,
csrc/mla_decode_a16w8_api.cpp:152-178, csrc/mla_decode_a16w8_multiq_api.cpp:177-196).
The library is loaded once; a missing or incomplete library raises ImportError
at import time -- there is no fallback path.
"""
import ctypes
import importlib
import os
import re
import warnings

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("MOONMATH_LIB") or os.path.join(_HERE, "libmoonmath_gfx950.so")

_p = ctypes.c_void_p
_i = ctypes.c_int
_f = ctypes.c_float
_sz = ctypes.c_size_t
_ip = ctypes.POINTER(ctypes.c_int)

# name -> (restype, argtypes)
SIGNATURES = {}
for _m in ("rtne", "rtna", "rtz"):
    SIGNATURES[f"launch_v_transpose_{_m}"] = (_i, [_p, _p, _i, _i, _i, _i, _p])
    SIGNATURES[f"launch_attention_forward_{_m}"] = (_i, [_p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _p, _p])
    SIGNATURES[f"tail_workspace_bytes_{_m}"] = (_sz, [])
    SIGNATURES[f"launch_attention_forward_lite_{_m}"] = (
        _i, [_p, _p, _p, _p, _i, _i, _i, _i, _i, _p, _p, _p, _f, _i, _i, _p, _p])
    SIGNATURES[f"lite_workspace_bytes_{_m}"] = (_sz, [_i, _i, _i])
SIGNATURES.update({
    "moonmath_attention_forward_ex": (_i, [_p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _i, _p]),
    "moonmath_attention_forward_direct": (_i, [_p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _p, _i, _p]),
    "moonmath_attention_forward_lite_direct": (
        _i, [_p, _p, _p, _p, _i, _i, _i, _i, _i, _p, _p, _p, _f, _i, _i, _i, _p, _p]),
    "moonmath_attention_direct_workspace": (_sz, [_i, _i, _i, _i]),
    "moonmath_attention_prefers_direct": (_i, [_i, _i, _i, _i]),
    "moonmath_attention_plan_tail": (_i, [_i, _i, _i, _i, _i, _i, _ip]),
    "moonmath_attention_geometry": (_i, [_ip]),
    "moonmath_attention_vt_bytes": (_sz, [_i, _i, _i]),
    # MLA decode (reference csrc/mla_decode_a16w8_api.cpp:19-33, multiq_api.cpp:22-34)
    "mla_decode_a16w8_workspace_bytes": (_sz, []),
    "mla_decode_a16w8_multiq_workspace_for": (_sz, [_i, _i, _i, _i]),
    "launch_mla_decode_a16w8": (_i, [_p, _p, _p, _p, _p, _i, _i, _i, _i, _i, _f, _f, _f, _p, _p]),
    "launch_mla_decode_a16w8_paged_dev": (
        _i, [_p, _p, _p, _p, _p, _p, _p, _p, _i, _i, _i, _i, _i, _f, _f, _f, _p, _p, _sz, _i]),
    "launch_mla_decode_a16w8_paged_dev_noalloc": (
        _i, [_p, _p, _p, _p, _p, _p, _p, _p, _i, _i, _i, _i, _i, _f, _f, _f, _p, _sz, _i]),
    "mla_decode_a16w8_blocks_index_bytes": (_sz, [_i, _i]),
    "launch_mla_decode_a16w8_paged_blocks_dev": (
        _i, [_p, _p, _p, _p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _i, _i, _f, _f, _f, _p, _p, _p]),
    "launch_mla_decode_a16w8_multiq": (_i, [_p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _f, _f, _p, _p]),
    "launch_mla_decode_a16w8_multiq_paged_dev": (
        _i, [_p, _p, _p, _p, _p, _p, _p, _p, _i, _i, _i, _i, _i, _i, _f, _f, _p, _p, _sz]),
    "mla_decode_a16w8_plan_parts": (_i, [_i, _i, _i, _i]),
    "mla_decode_a16w8_plan_parts_q": (_i, [_i, _i, _i, _i]),
    "mla_decode_a16w8_plan_parts_capped": (_i, [_i, _i, _i, _i]),
    "mla_decode_a16w8_multiq_plan_parts_q": (_i, [_i, _i, _i, _i]),
    "mla_decode_a16w8_max_ctas": (_i, []),
    "moonmath_mla_effective_parts": (_i, [_i, _i, _i, _i, _i]),
    "moonmath_mla_slab_parts": (_i, [_i, _i, _i, _i]),
    "moonmath_mla_split": (_i, [_i, _ip, _i, _i, _i, ctypes.c_longlong, _ip, _i]),
    "moonmath_fp8e4m3_to_bf16": (_i, [_p, _p, _i, _p]),
    "moonmath_pack_bf16": (_i, [_p, _p, _i, _i, _p]),
    "launch_mla_kv_quantize": (_i, [_p, _p, _p, _p, ctypes.c_longlong, ctypes.c_longlong, _f, _i, _p]),
})


class _Lib:
    def __init__(self, path):
        if not os.path.exists(path):
            raise ImportError(
                f"moonmath_attention: HIP library not found at {path}. "
                "Build it with `python amd-kernels_amd/build_lib.py` (hipcc, gfx950)."
            )
        self.path = path
        self.dll = ctypes.CDLL(path)
        missing = []
        for name, (res, args) in SIGNATURES.items():
            try:
                fn = getattr(self.dll, name)
            except AttributeError:
                missing.append(name)
                continue
            fn.restype = res
            fn.argtypes = args
            setattr(self, name, fn)
        if missing:
            raise ImportError(f"moonmath_attention: {path} lacks symbols {missing}; rebuild it")


lib = _Lib(LIB_PATH)

class _PythonOnly:
    """In the native path's place: leaves every call to the Python path."""

    def __getattr__(self, name):
        return lambda *args: None


def load_calls():
    """The native path of plain GPU calls (csrc/calls.cpp), bound to ``lib``'s
    launchers. It is compiled against one torch; with another the wrappers' Python
    path makes the same launches."""
    try:
        calls = importlib.import_module("._calls", __package__)
        built = calls.torch_version()
        if built != re.match(r"[\d.]*\d", torch.__version__).group():
            raise ImportError(f"built against torch {built}, running {torch.__version__}")
    except ImportError as e:
        warnings.warn(
            f"moonmath_attention: the _calls module is not usable ({e}): calls take ~10 us more on the host. "
            "Build it with `python amd-kernels_amd/build_lib.py`.", RuntimeWarning, stacklevel=2)
        return _PythonOnly()
    calls.bind({name: ctypes.cast(getattr(lib.dll, name), _p).value for name in calls.bound_names()})
    return calls


calls = load_calls()


def stream_ptr(device):
    """Raw hipStream_t of torch's current stream on ``device``."""
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(0)


def geometry():
    out = (ctypes.c_int * 4)()
    rc = lib.moonmath_attention_geometry(out)
    if rc != 0:
        raise RuntimeError(f"moonmath_attention_geometry returned {rc}")
    return {"rows_per_cta": out[0], "kv_block": out[1], "slots": out[2], "max_parts": out[3]}


def plan_tail(batch, heads, seq_len, seq_len_kv, enable=True, force_split_ways=0):
    out = (ctypes.c_int * 4)()
    rc = lib.moonmath_attention_plan_tail(batch, heads, seq_len, seq_len_kv, int(enable), force_split_ways, out)
    if rc != 0:
        raise ValueError(f"moonmath_attention_plan_tail returned {rc}")
    return tuple(out)
