"""Native forms of the wrappers' checks and calls (csrc/fast_call.cpp).

Each function takes a wrapper's arguments in order, and either makes the call and returns its result (a
launch that fails raises, as on the Python path) or returns None before the entry point launches anything:
the arguments are then for the checked Python path, which accepts more forms (array carriers, host values)
and raises the errors.  Without a usable extension every call takes that path, after one warning.
"""
from __future__ import annotations

import ctypes
import importlib.util
import os
import warnings

from .. import _capi

EXT_PATH = os.path.join(os.path.dirname(_capi.LIB_PATH), "_fast_call.so")
_NAMES = ("decode", "prep_decode", "prefill", "prep_prefill", "prep_append", "store", "store_layers")
# the C entry points the extension calls, in the order it takes their addresses
_ENTRIES = ("ifn_store_kv", "ifn_store_kv_layers", "ifn_paged_decode_workspace_bytes",
            "ifn_paged_decode_plan_bytes", "ifn_paged_decode",
            "ifn_paged_decode_append", "ifn_paged_decode_planned", "ifn_paged_decode_append_planned",
            "ifn_paged_decode_planning", "ifn_paged_decode_append_planning",
            "ifn_paged_decode_shared_prefix_workspace_bytes", "ifn_paged_decode_shared_prefix",
            "ifn_paged_prefill_workspace_bytes", "ifn_paged_prefill", "ifn_paged_prefill_append",
            "ifn_qk_norm_rope_append", "ifn_paged_decode_prep_append", "ifn_paged_decode_prep_append_planning",
            "ifn_paged_prefill_prep_append")


def _none(*args):
    return None


def _signature(name):
    res, args = _capi.SIGNATURES[name]
    return f"{name}:{''.join(t._type_ for t in (res, *args))},"


def load():
    """The extension, bound to the loaded library's entry points.

    ImportError when it was compiled for other entry points or signatures than ``_capi`` declares (ctypes'
    type letters, compared in ``bind``)."""
    lib = _capi.lib()
    spec = importlib.util.spec_from_file_location("_fast_call", EXT_PATH)
    ext = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(ext)
    ext.bind("".join(map(_signature, _ENTRIES)),
             *(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _ENTRIES))
    return ext


def _first(name):
    def call(*args):
        try:
            _capi.lib()
        except _capi.NativeLibraryError:
            return None  # (the Python path says what is missing)
        try:
            ext = load()
            globals().update({n: getattr(ext, n) for n in _NAMES})
        except Exception as e:  # missing, unloadable or stale: no reason to refuse a call
            globals().update(dict.fromkeys(_NAMES, _none))
            warnings.warn(f"{EXT_PATH}: {e}; the wrappers' checks run in Python", RuntimeWarning, stacklevel=3)
        return globals()[name](*args)
    return call


decode, prep_decode, prefill, prep_prefill, prep_append, store, store_layers = (_first(n) for n in _NAMES)
