"""The host library, loaded once per process: the cache manager's core and the samplers' uniform numbers."""
from __future__ import annotations

import ctypes

_lib = None


def host_library() -> ctypes.CDLL:
    """The library of csrc/host (built if it is not there), its functions' types declared."""
    global _lib
    if _lib is None:
        from . import build

        lib = ctypes.CDLL(build.ensure_host_built())
        if lib.egh_abi_version() != 5:
            raise RuntimeError("the host library has an unexpected ABI version")
        vp, i = ctypes.c_void_p, ctypes.c_int
        sigs = {
            "egh_create": ([i, vp, vp, i, i], vp), "egh_destroy": ([vp], None), "egh_set_keep_first": ([vp, i, i], i), "egh_admit": ([vp], i),
            "egh_release": ([vp, i], i), "egh_slot": ([vp, i], i), "egh_num_tokens": ([vp, i], i),
            "egh_version": ([vp, i], i), "egh_table_len": ([vp, i, i], i), "egh_table": ([vp, i, i, vp, i], i),
            "egh_pages_needed": ([vp, i, i, vp], i), "egh_free_pages": ([vp, i], i), "egh_used_pages": ([vp, i], i),
            "egh_num_pages": ([vp, i], i), "egh_high_water": ([vp, i], i), "egh_free_slots": ([vp], i),
            "egh_reserve": ([vp, i, vp, vp, vp], i), "egh_commit": ([vp, i, vp, vp], i), "egh_unreserve": ([vp, i, vp], i),
            "egh_slot_index": ([vp, i, i, i], i), "egh_check": ([vp, vp, i], i),
            "egh_fill_decode": ([vp, i, vp, vp, vp, vp, vp], i),
            "egh_fill_decode_rows": ([vp, i, i, vp, vp, vp, vp, vp], i),
            "egh_uniforms": ([i, vp, vp, vp, vp], None),
            "egh_fill_step": ([vp, i, vp, vp, vp, vp, vp, vp, vp, vp, vp, vp], i),
        }
        for name, (args, res) in sigs.items():
            fn = getattr(lib, name)
            fn.argtypes, fn.restype = args, res
        _lib = lib
    return _lib
