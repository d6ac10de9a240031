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


def _batch(n, seed):
    rng = np.random.Generator(np.random.Philox(seed))
    x = np.zeros((n, 32), dtype=np.float32)
    x[:, :18] = rng.normal(0, 1, (n, 18))
    return x, rng.normal(0, 1, (n, 8)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 257])
def test_gradient_at_tile_edges(dev, n):
    """The one-kernel gradient where a wavefront's 16 points and a tile's 128 end: against the CPU
    restatement, and against the forward and backward kernels called one after the other (the
    same bounds: both differ by roundings to bf16 that fall the other way)."""
    import ctypes
    from ice3_amd import _lib
    from ice3_amd import surrogate as S
    from ice3_amd._fields import ptr
    from oracle import mlp_oracle as mo
    p = S.init_params(13)
    p[mo.NW:mo.NW + 4 * 128] = np.random.Generator(np.random.Philox(6)).normal(0, 0.2, 4 * 128)
    mlp = S.MLP(device=0, params=p)
    x, t = _batch(n, 40 + n)
    xb, tt = torch.as_tensor(x).to(dev).to(torch.bfloat16), torch.as_tensor(t).to(dev)
    sse = mlp.gradient(xb, tt).item()
    fused = mlp.grad.cpu().numpy()
    loss, gr = mo.loss_and_grad(p, xb.float().cpu().numpy(), t, emulate=True)
    f32 = dict(dtype=torch.float32, device=dev)
    z, h, dy = torch.empty((4, n, 128), **f32), torch.empty((4, n, 128), dtype=torch.bfloat16, device=dev), \
        torch.empty((n, 32), **f32)
    lp, gp, g = torch.empty(-(-n // 128), **f32), torch.empty((-(-n // 128), S.sizes()["n_params"]), **f32), \
        torch.empty(S.sizes()["n_params"], **f32)
    sp = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    assert mlp.lib.ice3_mlp_forward(n, ptr(mlp.wpk), ptr(mlp.params), ptr(xb), ptr(tt), None, ptr(z), ptr(h),
                                    ptr(dy), ptr(lp), sp) == _lib.ICE3_OK
    assert mlp.lib.ice3_mlp_backward(n, ptr(mlp.wrm), ptr(xb), ptr(z), ptr(h), ptr(dy), ptr(gp), ptr(g),
                                     sp) == _lib.ICE3_OK
    for other, sse2 in ((gr, float(loss)), (g.cpu().numpy(), lp.sum().item())):
        assert abs(sse - sse2) <= 1e-3 * sse2
        o = 0
        for k, m in mo.DIMS + [(1, mo.NB)]:
            a, b = fused[o:o + k * m], other[o:o + k * m]
            assert np.linalg.norm(a - b) < 2e-2 * np.linalg.norm(b), (k, m)
            o += k * m
    assert np.all(fused[18 * 128:32 * 128] == 0)
    assert np.all(fused[mo.NW - 128 * 32:mo.NW].reshape(128, 32)[:, 8:] == 0)


@pytest.mark.parametrize("tiles", [1, 15, 16, 17, 33, 145])
def test_gradient_sums_every_partial(dev, tiles):
    """The sum over tiles (16 wavefronts, eight loads at a time) against a float64 sum of the
    same partials: an fp32 sum of m terms in any order is within m 2^-24 of the terms' magnitudes."""
    from ice3_amd import surrogate as S
    mlp = S.MLP(device=0, seed=14)
    x, t = _batch(tiles * 128 - 77, 60 + tiles)
    sse = mlp.gradient(torch.as_tensor(x).to(dev).to(torch.bfloat16), torch.as_tensor(t).to(dev)).item()
    part = mlp.gpart.double()
    assert part.shape[0] == tiles
    assert bool(((mlp.grad.double() - part.sum(0)).abs() <= tiles * 2.0 ** -24 * part.abs().sum(0)).all())
    lp = mlp.loss_part.double().sum().item()
    assert abs(sse - lp) <= (tiles + 64) * 2.0 ** -24 * lp


def test_gradient_refuses_an_unaligned_workspace(dev):
    """The partials are stored by 16 bytes."""
    import ctypes
    from ice3_amd import _lib
    from ice3_amd._fields import ptr
    lib = _lib.load()
    a = torch.zeros(1 << 17, dtype=torch.float32, device=dev)
    off = ctypes.c_void_p(a.data_ptr() + 4)
    assert lib.ice3_mlp_gradient(1, *[ptr(a)] * 5, off, *[ptr(a)] * 3, None) == _lib.ICE3_EINVAL
