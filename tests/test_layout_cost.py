"""What a call on arrays that need no copy costs on the host: bringing them to a kernel's order makes no
more tensors than as_columns of each would, and the order is settled by no more looks than it takes."""
import pytest

torch = pytest.importorskip("torch")

from torch.overrides import TorchFunctionMode  # noqa: E402

from ice3_amd import _fields as F  # noqa: E402
from ice3_amd.ice_adjust import IceAdjust  # noqa: E402

CPU = torch.device("cpu")
NAMES = ("th", "pabs", "rv", "rc", "ri", "rr", "rs", "rg", "exn")


class Tensors(TorchFunctionMode):
    """Counts the torch calls that return a tensor."""

    def __init__(self):
        super().__init__()
        self.made = 0

    def __torch_function__(self, func, types, args=(), kwargs=None):
        r = func(*args, **(kwargs or {}))
        self.made += isinstance(r, torch.Tensor)
        return r


def _fields(shape, order):
    rows = {k: torch.rand(shape, dtype=torch.float64) for k in NAMES}
    if order == "rows":
        return rows
    nz = shape[-1]
    return {k: v.reshape(-1, nz).t().contiguous().t().reshape(shape) for k, v in rows.items()}


def _of_each(f):
    with Tensors() as n:
        return {k: F.as_columns(v, "jax", device=CPU, name=k) for k, v in f.items()}, n.made


@pytest.mark.parametrize("shape", [(4, 5, 7), (1, 1, 2), (6, 3)])
def test_ice_adjust_takes_column_views_as_cheaply_as_each(shape):
    f = _fields(shape, "columns")
    ref, most = _of_each(f)
    call = IceAdjust.__new__(IceAdjust)
    call.device = CPU
    sq = torch.zeros(shape[:-1], dtype=torch.float64)
    with Tensors() as n:
        got, _, nlev, ncol, rows = call._inputs(sq, f, "jax")
    with Tensors() as per_column:
        call._per_column(sq, "sigqsat", ncol, "jax")
    assert n.made - per_column.made <= most
    for k, v in got.items():
        assert v.data_ptr() == f[k].data_ptr()  # no copy
        assert torch.equal(v.t() if rows else v, ref[k])


@pytest.mark.parametrize("shape,order", [((4, 5, 7), "columns"), ((1, 1, 2), "rows"), ((5, 1), "rows"), ((1, 9), "rows")])
def test_fields_in_order_are_taken_as_cheaply_as_each(shape, order):
    f = _fields(shape, order)
    ref, most = _of_each(f)
    with Tensors() as n:
        got, fresh = F.columns_of(f, "jax", device=CPU)
    assert n.made <= most and not fresh
    for k, v in got.items():
        assert v.data_ptr() == f[k].data_ptr() and torch.equal(v, ref[k])


@pytest.mark.parametrize("views", range(len(NAMES) + 1))
def test_order_is_settled_by_the_fewest_looks(views):
    """As many rows as views or more: rows, with no look at the views; more views: columns, after one
    look more than there are rows."""
    r, c = _fields((4, 5, 7), "rows"), _fields((4, 5, 7), "columns")
    f = {k: (c if q < views else r)[k] for q, k in enumerate(NAMES)}
    rows = len(NAMES) - views
    with Tensors() as n:
        assert F.in_rows(f) == (rows >= views)
    assert n.made == (0 if rows >= views else rows + 1)
