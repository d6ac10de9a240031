"""The statistical sedimentation's two forms on the GPU: k_sedim (a wavefront per 64 columns,
species and half, levels in groups) at the sizes where it can go wrong, its surface rates
against the oracle's, and the fused and mixed steps on both sides of the column count from
which one thread walks a column, every output bit for bit."""
import numpy as np
import pytest

from helpers import floor_for, rel_err

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 1e-11
DT = 50.0
KEYS = dict(exn="exn", dzz="dzz", rhodj="rhodj", rhodref="rhodref", exnref="exn_ref", pres="pabs", cf="cldfr",
            hlc_hrc="hlc_hrc", hlc_hcf="hlc_hcf", hli_hri="hli_hri", hli_hcf="hli_hcf", sigs="sigs", th_t="tht",
            rv_t="rvt", rc_t="rct", rr_t="rrt", ri_t="rit", rs_t="rst", rg_t="rgt", ci_t="ci", ths="ths",
            rvs="rvs", rcs="rcs", rrs="rrs", ris="ris", rss="rss", rgs="rgs")


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda", 0)


def _state(ncol, nlev, hail):
    """The pipeline profile's lowest nlev levels (every third one where 90 levels allow it)."""
    from ice3_amd import synthetic
    from oracle import oracle_lib, ref_lib
    f = synthetic.generate(ncol, 90, seed=20260300 + ncol + nlev, variant="pipeline")
    if hail:
        f["rh"] = f["rg"] * np.random.Generator(np.random.Philox(nlev)).uniform(0.2, 2.0, f["rg"].shape)
        f["rhs"] = f["rh"] / DT
    pick = slice(0, 3 * nlev, 3) if nlev <= 30 else slice(0, nlev)
    f = {k: np.ascontiguousarray(v[pick]) if v.ndim == 2 else v for k, v in f.items()}
    s = ref_lib.pipeline_state(f, (oracle_lib.ice_adjust_hail if hail else oracle_lib.ice_adjust)(f))
    s["ci"] = f["ci"]
    if hail:
        s["rht"], s["rhs"] = f["rhs"] * DT, f["rhs"]
    return s


@pytest.mark.parametrize("hail", [False, True])
@pytest.mark.parametrize("ncol,nlev", [(1, 1), (63, 2), (64, 3), (65, 4), (129, 7), (200, 90)])
def test_surface_rates_at_group_edges(dev, ncol, nlev, hail):
    from ice3_amd import RainIce, RainIceHail
    from oracle import oracle_lib
    s = _state(ncol, nlev, hail)
    st = {k: s[v] for k, v in KEYS.items()}
    if hail:
        st.update(rh_t=s["rht"], rhs=s["rhs"])
    _, diags = (RainIceHail if hail else RainIce)()(st, DT)
    ref = (oracle_lib.rain_ice_hail if hail else oracle_lib.rain_ice)(s, DT)
    for k in ("inprc", "inprr", "inpri", "inprs", "inprg") + (("inprh",) if hail else ()):
        assert rel_err(diags[k].cpu().numpy(), ref[k], floor_for(k, TOL)).max() <= TOL, k


@pytest.mark.parametrize("nlev", [2, 3, 7])
@pytest.mark.parametrize("kind", ["fp64", "mixed", "hail"])
def test_column_walk_and_split_form_agree(dev, kind, nlev):
    """One column more than the walk's threshold, against the same columns in two calls below
    it."""
    from ice3_amd import AdjustRainIce, AdjustRainIceHail, synthetic
    ncol = 432 * torch.cuda.get_device_properties(dev).multi_processor_count + 1
    f = synthetic.generate(ncol, nlev, seed=20260311, variant="pipeline")
    f["rhodref"] = f["rho_dry_ref"]
    f["rh"] = f["rg"] * 0.7
    f["rhs"] = f["rh"] / DT
    f = {k: torch.from_numpy(v).to(dev) for k, v in f.items()}
    call = AdjustRainIceHail() if kind == "hail" else AdjustRainIce()
    kw = {"precision": "mixed"} if kind == "mixed" else {}
    whole = call(f, DT, **kw)
    half = ncol // 2
    parts = [call({k: v[..., c].contiguous() for k, v in f.items()}, DT, **kw)
             for c in (slice(0, half), slice(half, ncol))]
    for k, v in whole.items():
        assert torch.equal(v, torch.cat([p[k] for p in parts], dim=-1)), k
