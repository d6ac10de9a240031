"""Which arrays RAIN_ICE takes: the entry with sources apart from what it writes refuses a source that
another output would overwrite."""
import ctypes
import re

import pytest

from ice3_amd import _lib

SRC = ("ths", "rvs", "rcs", "rrs", "ris", "rss", "rgs", "ci", "rhs")
SCALARS = ("evap3d", "rainfr", "inprc", "inprr", "inpri", "inprs", "inprg", "inprh")


def _from(alias_src, alias_out, prec="fp64", hail=True, ncol=4):
    """ice3_rain_ice_from with made-up addresses and a context of zeros (never followed: the call is
    refused), the source alias_src given the address of the output alias_out."""
    p = {}

    def addr(k):
        return p.setdefault(k, 4096 * (len(p) + 1))

    fin = _lib.RainIn(*[addr("in " + k) for k in _lib.RAIN_IN_FIELDS])
    src = {k: addr("src " + k) for k in SRC}
    io = {k: addr("io " + k) for k in SRC}
    out = {k: addr("out " + k) for k in SCALARS}
    src[alias_src] = io[alias_out] if alias_out in io else out[alias_out]
    csrc = _lib.RainSrc(*[src[k] for k in SRC])
    cio = _lib.RainIO(*[io[k] for k in SRC[:8]])
    cout = _lib.RainOut(*[out[k] for k in _lib.RAIN_OUT_FIELDS])
    h = _lib.Hail(addr("rht"), io["rhs"], out["inprh"]) if hail else None
    ctx = ctypes.create_string_buffer(1 << 20)
    return _lib.load().ice3_rain_ice_from(
        ctypes.cast(ctx, ctypes.c_void_p), _lib.PREC_FP64 if prec == "fp64" else _lib.PREC_MIXED, ncol, 3, 4, 50.0,
        ctypes.byref(fin), None, ctypes.byref(csrc), ctypes.byref(cio), ctypes.byref(cout),
        ctypes.byref(h) if h else None, None, None)


def test_source_struct_matches_header():
    import os
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    hdr = open(os.path.join(root, "include", "ice3.h")).read()
    body = re.search(r"typedef struct \{([^}]*)\} ice3_rain_ice_src;", hdr).group(1)
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    assert tuple(re.findall(r"\*\s*(\w+)", body)) == tuple(f for f, _ in _lib.RainSrc._fields_) == SRC


@pytest.mark.parametrize("source", SRC)
def test_crossed_sources_are_refused(source):
    """Every output but the source's own array, in both precisions."""
    for other in SRC + SCALARS:
        if other != source:
            assert _from(source, other) == _lib.ICE3_EINVAL, other
            if "rhs" not in (source, other) and other != "inprh":
                assert _from(source, other, prec="mixed", hail=False) == _lib.ICE3_EINVAL, other


def test_empty_domain_follows_no_pointer():
    assert _from("rrs", "rss", ncol=0) == _lib.ICE3_OK
