"""Which form the statistical sedimentation takes: one thread a column or several wavefronts for 64 of
them, and that no launch has 2^32 threads along an axis."""
import ctypes
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_stages"))
import host_lib  # noqa: E402

FORMS = {"fp64": 0, "hail": 1, "mixed": 2, "fused": 3}
DT = 50.0


@pytest.mark.parametrize("form", FORMS)
def test_several_threads_a_column_fit_a_launch(form):
    """A domain has at most 2^32 points (and a device far fewer than 4,096 compute units): the columns
    below the walk's count, at ten threads each, stay within a launch at every number of levels."""
    cols = host_lib.load().hst_sedim_walk_cols
    for nlev in [*range(1, 300), 1000, 65535]:
        most = min(cols(FORMS[form], nlev) * 4096, 2 ** 32 // nlev)
        assert 0 <= most and -(-most // 64) * 640 < 2 ** 32, nlev


def test_few_levels_walk_from_fewer_columns():
    cols = host_lib.load().hst_sedim_walk_cols
    for form in FORMS.values():
        counts = [cols(form, n) for n in range(1, 300)]
        assert counts[0] == 0                    # one level has nothing to wait for
        assert counts == sorted(counts) and counts[-1] <= 512


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


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "hail", "ocnd2", "mixed"])
@pytest.mark.parametrize("nlev", [1, 2, 3, 4, 7, 12, 40])
def test_rain_ice_on_both_sides_of_the_walk(kind, nlev):
    """RAIN_ICE over more columns than every form's walk begins at, against the same columns in calls of
    fewer than any walk of two levels or more: every output bit for bit (OCND2's model level height,
    the walk's and k_sedim's, through the microphysics that reads it)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ice3_amd import RainIce, RainIceHail, RainIceOCND2, synthetic
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    ncol, part = 512 * ncu + 1, 47 * ncu - 1
    f = synthetic.generate(2048, 90, seed=20260402, variant="pipeline")
    f = {k: np.ascontiguousarray(v[:3 * nlev:3] if nlev <= 30 else v[:nlev]) for k, v in f.items() if v.ndim == 2}
    rng = np.random.Generator(np.random.Philox(nlev))
    names = dict(exn="exn", rhodref="rho_dry_ref", pres="pabs", dzz="dzz", th_t="th", rv_t="rv", rc_t="rc", rr_t="rr",
                 ri_t="ri", rs_t="rs", rg_t="rg", ci_t="ci", sigs="sigs")
    names.update({k: k for k in ("ths", "rvs", "rcs", "rrs", "ris", "rss", "rgs")})
    s = {k: f[v] for k, v in names.items()}
    if kind == "hail":
        s["rh_t"], s["rhs"] = f["rg"] * 0.7, f["rg"] * 0.7 / DT
    if kind == "ocnd2":
        s.update(icldfr=rng.uniform(0, 1, f["th"].shape), ssio=rng.uniform(0, 0.2, f["th"].shape),
                 ssiu=rng.uniform(-0.2, 0, f["th"].shape), ifr=np.full(f["th"].shape, 10.0))
    # the columns over and over, thinned by as much as a column's own number says: none alike
    thin = torch.linspace(0.5, 1.5, ncol, dtype=torch.float64, device="cuda")
    s = {k: torch.from_numpy(v).cuda().repeat(1, -(-ncol // 2048))[:, :ncol].contiguous() for k, v in s.items()}
    for k in ("rrs", "ris", "rss", "rgs", "dzz") + (("rhs",) if kind == "hail" else ()):
        s[k] = s[k] * thin
    call = {"plain": RainIce, "hail": RainIceHail, "ocnd2": RainIceOCND2, "mixed": RainIce}[kind]()
    kw = {"precision": "mixed"} if kind == "mixed" else {}
    whole, whole_d = call(s, DT, **kw)
    for c in range(0, ncol, part):
        new, diags = call({k: v[:, c:c + part].contiguous() for k, v in s.items()}, DT, **kw)
        for k in ("ths", "rvs", "rcs", "rrs", "ris", "rss", "rgs", "ci_t", "evap3d") + (("rhs",) if kind == "hail" else ()):
            assert torch.equal(new[k], whole[k][:, c:c + part]), (k, c)
        for k in diags:
            assert torch.equal(diags[k], whole_d[k][c:c + part]), (k, c)


@pytest.mark.gpu
@pytest.mark.parametrize("hail", [False, True])
@pytest.mark.parametrize("nlev", [1, 2, 3, 4, 5])
def test_fused_step_of_few_levels(nlev, hail):
    """The fused step over more columns than its walk of any number of levels begins at, against the same
    columns in calls of fewer than its walk of three levels begins at (one and two levels are walked in
    both: ICE_ADJUST, the sedimentation and the microphysics one by one stand beside them)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ice3_amd import AdjustRainIce, AdjustRainIceHail, _lib, synthetic
    from ice3_amd._fields import ptr
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    ncol, part = 432 * ncu + 1, 143 * ncu - 1
    f = synthetic.generate(2048, 90, seed=20260404, variant="pipeline")
    f = {k: v[:3 * nlev:3] if v.ndim == 2 else v for k, v in f.items()}
    f["rhodref"] = f["rho_dry_ref"]
    f["rh"] = f["rg"] * 0.7
    f["rhs"] = f["rh"] / DT
    f = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in f.items()}
    f = {k: v.repeat((1,) * (v.dim() - 1) + (-(-ncol // 2048),))[..., :ncol].contiguous() for k, v in f.items()}
    for k in ("rrs", "ris", "rss", "rgs", "dzz"):
        f[k] = f[k] * torch.linspace(0.5, 1.5, ncol, dtype=torch.float64, device="cuda")
    call = AdjustRainIceHail() if hail else AdjustRainIce()
    whole = call(f, DT)
    for c in range(0, ncol, part):
        res = call({k: v[..., c:c + part].contiguous() for k, v in f.items()}, DT)
        for k, v in res.items():
            assert torch.equal(v, whole[k][..., c:c + part]), (k, c)
    if hail:
        return
    out = {k: torch.empty((nlev, ncol), dtype=torch.float64, device="cuda") for k in _lib.PIPE_OUT_FIELDS[:15]}
    out.update({k: torch.empty(ncol, dtype=torch.float64, device="cuda") for k in _lib.PIPE_OUT_FIELDS[15:]})
    fin = _lib.PipeIn(*[ptr(f[k]) for k in _lib.PIPE_IN_FIELDS])
    fout = _lib.PipeOut(*[ptr(out[k]) for k in _lib.PIPE_OUT_FIELDS])
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for stage in (_lib.STAGE_ADJUST, _lib.STAGE_SEDIMENTATION, _lib.STAGE_MICROPHYSICS):
        assert _lib.load().ice3_adjust_rain_ice_stages(_lib.context(0), _lib.PREC_FP64, ncol, nlev, ncol, DT,
                                                       ctypes.byref(fin), ctypes.byref(fout), None, stage,
                                                       stream) == _lib.ICE3_OK
    for k, v in out.items():
        assert torch.equal(v, whole[k]), k
