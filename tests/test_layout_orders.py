"""The "jax" layout's memory orders: which order a call takes its fields in (CPU), and that ICE_ADJUST on
the arrays as they are gives the columns call's results bit for bit in every mix of orders (GPU)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ice3_amd._fields import as_columns, as_rows, in_rows  # noqa: E402

DT = 50.0
ARGS = ("pabs", "sigs", "th", "exn", "exn_ref", "rho_dry_ref", "rv", "rc", "ri", "rr", "rs", "rg",
        "cf_mf", "rc_mf", "ri_mf", "rvs", "rcs", "ris", "ths")


def _column_view(rows):
    """A (nx, ny, nz) view whose memory is (nz, nx * ny), as a columns call's results are."""
    nz = rows.shape[-1]
    return rows.reshape(-1, nz).t().contiguous().t().reshape(rows.shape)


@pytest.mark.parametrize("shape", [(3, 5, 7), (1, 1, 4), (2, 3, 1), (6, 4), (2, 2, 3, 5)])
def test_orders_hold_the_same_field(shape):
    t = torch.arange(float(np.prod(shape)), dtype=torch.float64).reshape(shape)
    forms = {"rows": t, "columns": _column_view(t), "strided": torch.stack([t, t], -1)[..., 0],
             "first axis last": t.movedim(0, -1).contiguous().movedim(-1, 0)}
    for name, x in forms.items():
        assert torch.equal(x, t), name
        assert torch.equal(as_rows(x, name), t.reshape(-1, shape[-1])), name
        assert as_rows(x, name).is_contiguous()
        assert torch.equal(as_columns(x, "jax", device="cpu", name=name), t.reshape(-1, shape[-1]).t()), name


def test_order_of_a_call():
    t = torch.zeros((3, 5, 7), dtype=torch.float64)
    c = _column_view(t)
    s = torch.stack([t, t], -1)[..., 0]
    assert in_rows({"a": t, "b": t})
    assert not in_rows({"a": c, "b": c, "c": t})
    assert in_rows({"a": c, "b": t})
    assert in_rows({"a": s})  # neither order: a copy either way
    with pytest.raises(ValueError):
        as_rows(torch.zeros(3, dtype=torch.float64), "a")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "hail", "ocnd2"])
@pytest.mark.parametrize("shape", [(1, 1, 2), (3, 7, 5), (5, 13, 90), (16, 16, 17)])
def test_ice_adjust_orders_bitwise(kind, shape):
    from ice3_amd import IceAdjust, IceAdjustHail, IceAdjustOCND2, synthetic
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    nx, ny, nz = shape
    rng = np.random.Generator(np.random.Philox(nz))
    f = synthetic.generate(nx * ny, nz, seed=20260320 + nz, variant="pipeline")
    f["cf_mf"] = rng.uniform(0.0, 0.3, f["th"].shape)
    f["rc_mf"], f["ri_mf"] = f["cf_mf"] * 1e-5, f["cf_mf"] * 2e-5
    extra = {}
    if kind == "hail":
        extra = {"rh": f["rg"] * 0.7}
    if kind == "ocnd2":
        extra = {"zz": np.broadcast_to(synthetic.level_profile(nz)[2][:, None], f["th"].shape) + f["sigs"],
                 "ice_cld_wgt": rng.uniform(0.5, 1.5, nx * ny)}
    call = {"plain": IceAdjust, "hail": IceAdjustHail, "ocnd2": IceAdjustOCND2}[kind]()
    sq = torch.from_numpy(rng.uniform(0.01, 0.03, nx * ny)).cuda()
    cols = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in {**{k: f[k] for k in ARGS}, **extra}.items()}

    def run(to):
        x = {k: to(k, v) if v.dim() == 2 else v for k, v in cols.items()}
        return call(sq, *[x[k] for k in ARGS], timestep=DT, return_srcs=True, **{k: x[k] for k in extra})

    ref = run(lambda k, v: v)
    rows = lambda k, v: v.t().contiguous().reshape(shape)  # noqa: E731
    view = lambda k, v: v.t().reshape(shape)  # noqa: E731
    orders = {"rows": rows, "columns": view,
              "mostly rows": lambda k, v: (view if k in ("rv", "ths") else rows)(k, v),
              "mostly columns": lambda k, v: (rows if k in ("rv", "ths", "zz") else view)(k, v),
              "strided": lambda k, v: torch.stack([rows(k, v)] * 2, -1)[..., 0]}
    for name, to in orders.items():
        res = run(to)
        for r, e in zip(res, ref):
            assert r.shape == shape
            assert torch.equal(r.reshape(-1, nz).t().nan_to_num(7.0), e.nan_to_num(7.0)), name
    bad = {k: rows(k, v).clone() if v.dim() == 2 else v for k, v in cols.items()}
    bad["rc"][0, 0, 0] = float("nan")
    with pytest.raises(ValueError, match=r"rc \(1\)"):
        call(sq, *[bad[k] for k in ARGS], timestep=DT, check_inputs=True, **{k: bad[k] for k in extra})


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(2, 2), (31, 5), (32, 128), (33, 129), (1000, 90), (65, 300), (300, 2)])
def test_transposing_launch(rows, cols):
    """Every field of a call in one launch: tile edges, more than one column tile, a field that needs no
    transposing among them."""
    from ice3_amd._fields import columns_of
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    t = {f"f{q}": torch.rand((rows, cols), dtype=torch.float64, device="cuda").reshape(1, rows, cols) for q in range(3)}
    t["view"] = _column_view(t["f0"])
    out, fresh = columns_of(t, "jax", device=torch.device("cuda", 0))
    assert list(out) == list(t) and fresh == {"f0", "f1", "f2"}
    for k, v in out.items():
        assert v.is_contiguous() and torch.equal(v, t[k].reshape(rows, cols).t()), k


@pytest.mark.gpu
@pytest.mark.parametrize("sedimentation", ["STAT", "SPLI"])
@pytest.mark.parametrize("kind", ["plain", "hail", "ocnd2"])
def test_rain_ice_orders_bitwise(kind, sedimentation):
    """RainIce in every order of its state, against the columns call; the caller's arrays stay as they were."""
    from ice3_amd import RainIce, RainIceHail, RainIceOCND2, synthetic
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    shape = (5, 13, 40)
    f = synthetic.generate(65, 40, seed=20260330, variant="pipeline")
    names = dict(exn="exn", exnref="exn_ref", rhodref="rho_dry_ref", rhodj="rhodj", pres="pabs", dzz="dzz",
                 th_t="th", rv_t="rv", rc_t="rc", rr_t="rr", ri_t="ri", rs_t="rs", rg_t="rg", ci_t="ci", sigs="sigs")
    names.update({k: k for k in ("ths", "rvs", "rcs", "rrs", "ris", "rss", "rgs")})
    cols = {k: f[v] for k, v in names.items()}
    cols["cf"] = (f["rc"] > 0) * 0.5
    if kind == "hail":
        cols["rh_t"], cols["rhs"] = f["rg"] * 0.7, f["rg"] * 0.7 / DT
    if kind == "ocnd2":
        rng = np.random.Generator(np.random.Philox(5))
        cols.update(icldfr=rng.uniform(0, 1, f["th"].shape), ssio=rng.uniform(0, 0.2, f["th"].shape),
                    ssiu=rng.uniform(-0.2, 0, f["th"].shape), ifr=np.full(f["th"].shape, 10.0))
    cols = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in cols.items()}
    call = {"plain": RainIce, "hail": RainIceHail, "ocnd2": RainIceOCND2}[kind](sedimentation=sedimentation)
    rows = lambda k, v: v.t().contiguous().reshape(shape)  # noqa: E731
    view = lambda k, v: v.t().reshape(shape)  # noqa: E731
    ref, ref_d = call(cols, DT)
    keys = ["ths", "rvs", "rcs", "rrs", "ris", "rss", "rgs", "ci_t", "evap3d", "rainfr"] + ["rhs"] * (kind == "hail")
    orders = {"rows": rows, "columns": view, "mixed": lambda k, v: (view if k in ("ths", "rv_t", "ci_t") else rows)(k, v)}
    for name, to in orders.items():
        state = {k: to(k, v.clone()) for k, v in cols.items()}
        new, diags = call(state, DT)
        for k in keys:
            assert new[k].shape == shape and torch.equal(new[k].reshape(65, 40).t(), ref[k]), (name, k)
        for k in ref_d:
            assert torch.equal(diags[k].reshape(-1), ref_d[k]), (name, k)
        for k, v in state.items():
            assert torch.equal(v.reshape(65, 40).t(), cols[k]), (name, k)
