"""The launchers' rules (fracture_amd/csrc/launch_rules.h) through their host build."""
import ctypes as C
from pathlib import Path

import pytest

_LIB = None


def lib():
    global _LIB
    if _LIB is None:
        path = Path(__file__).resolve().parents[1] / "fracture_amd" / "libfracture_hip_index.so"
        if not path.exists():
            pytest.fail(f"{path} is missing: run __graft_entry__.build()")
        _LIB = C.CDLL(str(path))
        _LIB.fhip_rule_paged_waves.argtypes = [C.c_int64, C.c_int, C.c_int]
        _LIB.fhip_rule_tq_route.argtypes = [C.c_int] * 9 + [C.c_int64, C.c_void_p]
        _LIB.fhip_rule_tq_route.restype = C.c_int64
        _LIB.fhip_rule_tq_workspace.argtypes = [C.c_int] * 4
        _LIB.fhip_rule_tq_workspace.restype = C.c_int64
        _LIB.fhip_rule_prefill_split.argtypes = [C.c_int] * 5 + [C.c_int64, C.c_int, C.c_int, C.c_void_p]
        _LIB.fhip_rule_prefill_split.restype = None
        _LIB.fhip_rule_prefill_fold.argtypes = [C.c_int, C.c_int64, C.c_int, C.c_int]
        _LIB.fhip_idx_prefill_code_offset.restype = C.c_uint32
    return _LIB


def paged_waves(queries, qh, kvh, hd, max_tokens, tok=1):
    """Waves per 1024-position split of an FP16 decode launch over tables of max_tokens positions."""
    heads = (qh // kvh + 7) // 8
    items = -(-queries // tok) * kvh * heads * max(1, -(-max_tokens // 1024))
    return lib().fhip_rule_paged_waves(items, hd, max_tokens)


VALU, DECODE, PREFILL = 0, 1, 2


class TqRoute:
    """Route of a TurboQuant attention call: kind, part (positions per partial), waves, tok (queries per
    workgroup), nsplit, split_pos, and bytes of the workspace that its layout takes."""

    def __init__(self, queries, qh, kvh, kbits, vbits, kv_len, causal=False, hd=128, ws_bytes=None):
        tokens = max(1, -(-kv_len // 16)) * 16
        if ws_bytes is None:
            ws_bytes = tq_workspace(queries, qh, hd, tokens)
        out = (C.c_int32 * 6)()
        self.bytes = lib().fhip_rule_tq_route(queries, qh, kvh, hd, kbits, vbits, tokens, kv_len, causal, ws_bytes, out)
        self.kind, self.part, self.waves, self.tok, self.nsplit, self.split_pos = out


def tq_workspace(queries, qh, hd, max_tokens):
    return lib().fhip_rule_tq_workspace(queries, qh, hd, max_tokens)


def prefill_split(queries, G, kvh, extent, max_splits):
    """Queries per block, blocks, splits, positions per split and workgroups of a tiled prefill."""
    out = (C.c_int64 * 5)()
    lib().fhip_rule_prefill_split(queries, G, kvh, 128, 64, 512, extent, max_splits, out)
    return tuple(out)
