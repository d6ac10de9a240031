"""The OCND2 branch's tabulated functions of temperature: every temperature, a NaN or an infinity too, has
an entry of the table."""
import ctypes
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_stages"))
import host_lib  # noqa: E402


def test_every_temperature_has_an_entry():
    lib = host_lib.load()
    lib.hst_tiwmx_index.argtypes = [ctypes.c_double]
    n = lib.hst_tiwmx_n()
    index = {t: lib.hst_tiwmx_index(t) for t in (-1e300, -np.inf, 0.0, 131.99, 132.0, 273.16, 373.16, 373.17, 1e300, np.inf)}
    assert index == {-1e300: 0, -np.inf: 0, 0.0: 0, 131.99: 0, 132.0: 0, 273.16: 14116, 373.16: n - 1, 373.17: n - 1,
                     1e300: n - 1, np.inf: n - 1}
    assert 0 <= lib.hst_tiwmx_index(np.nan) < n
