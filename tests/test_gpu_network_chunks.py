"""The surrogate step's network stage beyond a wavefront's first chunk: its rows in LDS used again and its
workgroup's queue appended to again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

WAVES, CHUNK, BLOCKS = 12, 64, 256  # wavefronts a workgroup, points a chunk, workgroups at most


def test_later_chunks_bitwise():
    """More than two chunks a wavefront, the last one ragged, against the same columns in calls of one
    chunk a wavefront at most: every output bit for bit, and each reason's count the sum of the parts'."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ice3_amd import surrogate as S
    from ice3_amd import synthetic
    first = WAVES * CHUNK * min(BLOCKS, torch.cuda.get_device_properties(0).multi_processor_count)
    nlev = 90
    ncol, part = (2 * first + first // 2) // nlev | 1, first // nlev
    assert ncol * nlev > 2 * first and ncol * nlev % CHUNK and part * nlev <= first
    f = synthetic.generate(ncol, nlev, seed=20260403, variant="pipeline")
    f["rhodref"] = f["rho_dry_ref"]
    f = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in f.items()}
    call = S.AdjustRainIceSurrogate(S.TrainedSurrogate.load())
    whole = call(f, 50.0, return_calls=True)
    count = call.last_counters
    assert count["network"] > 0 and count["network"] < ncol * nlev
    total = dict.fromkeys(count, 0)
    for c in range(0, ncol, part):
        res = call({k: v[..., c:c + part].contiguous() for k, v in f.items()}, 50.0, return_calls=True)
        for k, n in call.last_counters.items():
            total[k] += n
        for k, v in res.items():
            assert torch.equal(v, whole[k][..., c:c + part]), (k, c)
    assert total == count
