"""The persistent microphysics kernel's two orders of 64-point chunks (spread over the compute
units where the chunks are few, a workgroup's in a row where they are many): a domain just
past the change, ragged in its last chunk, against its two halves, every output bit for bit.
Points that outlast their chunk's own soft pass are parked among different neighbours in each."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DT = 50.0


@pytest.mark.parametrize("kind", ["fp64", "mixed", "ocnd2", "hail"])
def test_chunk_orders_agree(kind):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ice3_amd import AdjustRainIce, AdjustRainIceHail, AdjustRainIceOCND2, synthetic
    dev = torch.device("cuda", 0)
    nlev = 12
    chunks = 4 * torch.cuda.get_device_properties(dev).multi_processor_count * (12 if kind == "mixed" else 8)
    ncol = 64 * -(-chunks // nlev) - 63      # the fewest columns past the change
    f = synthetic.generate(ncol, nlev, seed=20260321, variant="pipeline")
    f["rhodref"] = f["rho_dry_ref"]
    if kind == "hail":
        f["rh"] = f["rg"] * 0.7
        f["rhs"] = f["rh"] / DT
    if kind == "ocnd2":
        f["zz"] = np.ascontiguousarray(np.broadcast_to(synthetic.level_profile(nlev)[2][:, None], f["th"].shape))
        f["ice_cld_wgt"] = np.full(ncol, 1.25)
    f = {k: torch.from_numpy(v).to(dev) for k, v in f.items()}
    call = {"ocnd2": AdjustRainIceOCND2, "hail": AdjustRainIceHail}.get(kind, AdjustRainIce)()
    kw = {"precision": "mixed"} if kind == "mixed" else {}
    whole = call(f, DT, return_calls=True, **kw)
    assert int((whole["calls"] > 2).sum()) > 1000
    half = ncol // 2 + 5
    parts = [call({k: v[..., c].contiguous() for k, v in f.items()}, DT, return_calls=True, **kw)
             for c in (slice(0, half), slice(half, ncol))]
    for k, v in whole.items():
        both = torch.cat([p[k] for p in parts], dim=-1)
        assert torch.equal(torch.nan_to_num(v, nan=1.0), torch.nan_to_num(both, nan=1.0)), k
