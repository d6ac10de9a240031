"""Launches of several threads a column: a launch takes fewer than 2^32 threads along an axis, so that
many columns go in parts."""
import ctypes
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_stages"))
import host_lib  # noqa: E402


@pytest.mark.parametrize("ncol", [1, 2 ** 28 - 1, 2 ** 28, 2 ** 28 + 1, 2 ** 29 + 65, 2 ** 31 - 1])
@pytest.mark.parametrize("hail", [False, True])
def test_sedimentation_in_parts_covers_every_column(ncol, hail):
    """Parts of whole workgroups' columns, each within a launch, one after the other, and every array
    of a part from its first column on (hail's seven arrays apart from the others')."""
    lib = host_lib.load()
    most = lib.hst_sedim_launch_cols()
    assert most % 64 == 0 and most // 64 * 640 < 2 ** 32
    arrays = [0 if q in (6, 11, 17) and not hail else (q + 1) << 40 for q in range(19)]
    given, part, c = (ctypes.c_size_t * 19)(*arrays), (ctypes.c_size_t * 19)(), 0
    while c < ncol:
        n = lib.hst_sedim_columns(ncol, c, most, given, part)
        assert 0 < n == min(most, ncol - c)
        assert list(part) == [a and a + 8 * c for a in arrays]
        c += n
    assert c == ncol


@pytest.mark.parametrize("rows,cols", [(2 ** 29, 2), (2 ** 31 - 1, 2), (2, 2 ** 31 - 1), (2 ** 24, 4096)])
def test_transposing_launch_refuses_more_tiles_than_it_takes(rows, cols):
    from ice3_amd import _lib
    p = (ctypes.c_void_p * 1)
    assert _lib.load().ice3_transpose_fields(1, p(4096), p(8192), rows, cols, None) == _lib.ICE3_EINVAL


@pytest.mark.gpu
@pytest.mark.parametrize("ncol", [2 ** 29 + 65])
def test_rain_ice_over_more_columns_than_one_axis_takes(ncol):
    """RAIN_ICE over one level of 2^29 + 65 columns (512 threads each 64) against the same columns among
    4,096: the profile's 4,096 points over and over."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    if torch.cuda.mem_get_info(0)[0] < 170e9:
        pytest.skip("needs 170 GB of GPU memory")
    from ice3_amd import RainIce, synthetic
    n = 4096
    f = synthetic.generate(n, 90, seed=20260401, variant="pipeline")
    f = {k: v[45:46] for k, v in f.items() if v.ndim == 2}  # a level with water and ice
    small = {k: torch.tensor(v, dtype=torch.float64, device="cuda") for k, v in {
        "exn": f["exn"], "dzz": f["dzz"], "rhodref": f["rho_dry_ref"], "pres": f["pabs"], "th_t": f["th"],
        "rv_t": f["rv"], "rc_t": f["rc"], "ri_t": f["ri"], "rr_t": f["rr"], "ci_t": f["ci"], "ths": f["ths"],
        "rvs": f["rvs"], "rcs": f["rcs"], "ris": f["ris"], "rrs": f["rrs"]}.items()}
    big = {k: v.repeat(1, ncol // n + 1)[:, :ncol].contiguous() for k, v in small.items()}
    for s in (small, big):  # snow and graupel share rain's arrays: 160 GB in all
        s.update(rs_t=s["rr_t"], rg_t=s["rr_t"], rss=s["rrs"], rgs=s["rrs"])
    ref, ref_d = RainIce()(small, 50.0)
    out, diags = RainIce()(big, 50.0)
    for got, want in ((out, ref), (diags, ref_d)):
        for k in got:
            if got[k] is not big.get(k):
                g, w = got[k].reshape(-1), want[k].reshape(-1)
                assert bool((g[:ncol // n * n].view(-1, n) == w).all()) and torch.equal(g[ncol // n * n:], w[:ncol % n]), k
    assert float(diags["inprr"].max()) > 0
