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
