"""The launchers' rules (fracture_amd/csrc/attn_rules.h) through their host build."""
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
    return _LIB


def paged_waves(queries, qh, kvh, hd, max_tokens, tok=1):
    """Waves per 1024-position split of an FP16 decode launch over tables of max_tokens positions."""
    heads = (qh // kvh + 7) // 8
    items = -(-queries // tok) * kvh * heads * max(1, -(-max_tokens // 1024))
    return lib().fhip_rule_paged_waves(items, hd, max_tokens)
