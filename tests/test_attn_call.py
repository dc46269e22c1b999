"""hx_varlen_attn_call's packed arguments, checked on the host before anything is launched."""

from __future__ import annotations

import ctypes
import re

import pytest

from helios_amd import _capi


def _fields():
    """Names of hx_attn_call's fields in order, from the header."""
    text = re.sub(r"/\*.*?\*/", "", _capi.HEADER_PATH.read_text(), flags=re.S)
    body = re.search(r"typedef struct hx_attn_call \{(.*?)\} hx_attn_call;", text, flags=re.S).group(1)
    names = []
    for line in body.split(";"):
        names += [part.split()[-1].lstrip("*") for part in line.split(",") if part.split()]
    return names


def _pack(**values):
    return _capi.ATTN_CALL.pack(*[values.get(n, 0) for n in _fields()])


def test_packed_struct_matches_the_header():
    names = _fields()
    assert names[0] == "size" and names.index("scale") == 19 and len(names) == 40
    assert _capi.ATTN_CALL.size == 8 * len(names)


@pytest.mark.parametrize("bad", [dict(size=0), dict(size=312), dict(batch=1 << 31), dict(max_q=-(1 << 40)),
                                 dict(workspace_bytes=-1), dict(head_dim=4), dict(n_q_heads=3, n_kv_heads=2)])
def test_bad_fields_are_refused(bad):
    good = dict(size=_capi.ATTN_CALL.size, batch=1, total_q=1, max_q=1, max_k=1, n_q_heads=2, n_kv_heads=2,
                head_dim=128, scale=1.0)
    lib = _capi.lib()
    code = lib.hx_varlen_attn_call(_pack(**{**good, **bad}), None)
    assert code in (_capi.HX_E_INVALID_ARG, _capi.HX_E_UNSUPPORTED)
    # with every field in range: refused for its null tensors, nothing launched
    assert lib.hx_varlen_attn_call(_pack(**good), None) == _capi.HX_E_INVALID_ARG
    assert lib.hx_varlen_attn_call(None, None) == _capi.HX_E_INVALID_ARG
    assert ctypes.sizeof(ctypes.c_int64) * 40 == _capi.ATTN_CALL.size
