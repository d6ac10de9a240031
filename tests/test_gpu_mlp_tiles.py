"""The matrix-core kernels at the sizes where their tiles end: a point's result does not depend on
the tile it falls in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda", 0)


@pytest.mark.parametrize("nlev,ncol", [(2, 1), (5, 3), (3, 11), (90, 1), (7, 37), (64, 64)])
def test_surrogate_step_tiles_bitwise(dev, nlev, ncol):
    """The surrogate step of ncol columns, network tiles of 32 points cut anywhere, against the same
    columns among 500."""
    from ice3_amd import surrogate as S
    from ice3_amd import synthetic
    f = synthetic.generate(500, nlev, seed=20260340 + nlev, variant="pipeline")
    f["rhodref"] = f["rho_dry_ref"]
    f = {k: torch.from_numpy(np.ascontiguousarray(v)).to(dev) for k, v in f.items()}
    call = S.AdjustRainIceSurrogate(S.TrainedSurrogate.load())
    whole = call(f, 50.0)
    part = call({k: v[..., 100:100 + ncol].contiguous() for k, v in f.items()}, 50.0)
    assert call.last_counters["network"] > 0 or ncol * nlev < 64
    for k, v in part.items():
        assert torch.equal(v, whole[k][..., 100:100 + ncol]), k
