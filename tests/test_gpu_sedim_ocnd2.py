"""RAIN_ICE with OCND2 where k_sedim's groups of three levels and of 64 columns end: its model level
height, which the microphysics reads, and the sedimentation, against the oracle."""
import numpy as np
import pytest

from helpers import cancellation_residuals, check_with_flips, explained_flips

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TOL = 1e-11
DT = 50.0
OUT = ("ths", "rvs", "rcs", "rrs", "ris", "rss", "rgs", "ci", "evap3d", "rainfr", "inprc", "inprr", "inpri",
       "inprs", "inprg")
KEYS = dict(exn="exn", dzz="dzz", rhodj="rhodj", rhodref="rhodref", exnref="exn_ref", pres="pabs", cf="cldfr",
            sigs="sigs", th_t="tht", rv_t="rvt", rc_t="rct", rr_t="rrt", ri_t="rit", rs_t="rst", rg_t="rgt", ci_t="ci",
            ths="ths", rvs="rvs", rcs="rcs", rrs="rrs", ris="ris", rss="rss", rgs="rgs", icldfr="icldfr", ssio="ssio",
            ssiu="ssiu", ifr="ifr")


@pytest.mark.parametrize("ncol", [63, 65, 1025])
@pytest.mark.parametrize("nlev", [2, 3, 4, 7, 8])
def test_sources_and_rates_at_group_edges(ncol, nlev):
    """Levels of the profile between +10 and -40 C, where the height reduces the nucleation.  At most
    six points (or 0.2 %, the bound elsewhere) may take another branch than the oracle, each shown to be
    one (helpers.explained_flips)."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ice3_amd import RainIceOCND2, synthetic
    from oracle import oracle_lib, ref_lib
    f = synthetic.generate(ncol, 90, seed=20260410 + ncol, variant="pipeline")
    f["zz"] = np.broadcast_to(synthetic.level_profile(90)[2][:, None], f["th"].shape)
    pick = np.linspace(1, 20, nlev).astype(int)
    f = {k: np.ascontiguousarray(v[pick]) if v.ndim == 2 else v for k, v in f.items()}
    f["ice_cld_wgt"] = np.random.Generator(np.random.Philox(ncol)).uniform(0.5, 1.5, ncol)
    s = ref_lib.pipeline_state_ocnd2(f, oracle_lib.ice_adjust_ocnd2(f))
    ref = oracle_lib.rain_ice_ocnd2(s, DT, with_iters=True)
    new, diags = RainIceOCND2()({k: s[v] for k, v in KEYS.items()}, DT, return_calls=True)
    out = {k: new["ci_t" if k == "ci" else k].cpu().numpy() for k in OUT[:10]}
    out.update({k: v.cpu().numpy() for k, v in diags.items()})
    run = lambda x: oracle_lib.rain_ice_ocnd2(x, DT, with_iters=True)  # noqa: E731
    flips = explained_flips(out, ref, run, s, OUT, TOL, ("tht", "rvt", "rct", "rrt", "rit", "rst", "rgt", "rvs", "rcs",
                                                         "rrs", "ris", "rss", "rgs", "ths"))
    flips |= cancellation_residuals(out, ref, s, OUT, TOL, DT)
    few = max(2e-3, 6 / flips.size)
    worst, nf, nb = check_with_flips(out, ref, OUT, flips, TOL, max_bad=few, max_flips=1.0)
    print(f"OCND2 {ncol}x{nlev}: {nf} flips, {nb} divergent of {flips.size}, worst {max(worst.values()):.1e}")
