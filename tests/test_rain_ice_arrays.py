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


UNREADABLE = {
    "objects": lambda np, torch: np.full((3, 4), None, dtype=object),
    "texts": lambda np, torch: np.full((3, 4), "1.0"),
    "byte order": lambda np, torch: np.zeros((3, 4), dtype=">f8"),
    "negative strides": lambda np, torch: np.zeros((3, 4))[::-1],
    "no data": lambda np, torch: torch.zeros((3, 4), dtype=torch.float64, device="meta"),
    "sparse": lambda np, torch: torch.zeros((3, 4), dtype=torch.float64).to_sparse(),
    "ragged": lambda np, torch: [[0.0, 1.0], [0.0]],
    "nothing": lambda np, torch: None,
}
READABLE = {
    "tensor": lambda np, torch: torch.zeros((3, 4), dtype=torch.float64),
    "single": lambda np, torch: torch.zeros((3, 4)),
    "view": lambda np, torch: torch.zeros((4, 3), dtype=torch.float64).t(),
    "array": lambda np, torch: np.zeros((3, 4), dtype=np.float32),
    "integers": lambda np, torch: np.zeros((3, 4), dtype=np.int64),
    "lists": lambda np, torch: [[0.0] * 4] * 3,
}


@pytest.mark.parametrize("layout", ["columns", "jax"])
@pytest.mark.parametrize("form", [*UNREADABLE, *READABLE])
def test_unread_fields_are_taken_and_refused_as_read_ones(form, layout):
    """A field that the interface takes and no kernel reads (rhodj): its shape alone is looked at, and
    it is refused where a field that is read would be."""
    import numpy as np
    import torch
    from ice3_amd._fields import as_columns, column_shape
    x = {**UNREADABLE, **READABLE}[form](np, torch)
    if form in READABLE:
        assert column_shape(x, layout, "x", device="cpu") == tuple(as_columns(x, layout, device="cpu", name="x").shape)
        return
    with pytest.raises(Exception) as read:
        t = as_columns(x, layout, device="cpu", name="x")
        t.data_ptr()  # what the call does with a field that it reads
    with pytest.raises(read.type):
        column_shape(x, layout, "x", device="cpu")


@pytest.mark.parametrize("shape,layout", [((3,), "columns"), ((3,), "jax"), ((2, 3, 4), "columns")])
def test_unread_fields_of_another_rank_are_refused(shape, layout):
    import numpy as np
    import torch
    from ice3_amd._fields import column_shape
    for x in (np.zeros(shape), torch.zeros(shape)):
        with pytest.raises(ValueError, match="x: expected"):
            column_shape(x, layout, "x", device="cpu")
