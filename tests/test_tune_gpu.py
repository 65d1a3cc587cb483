"""The tile autotuner (flashx_amd/tune.py) on given times."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ms,want", [((0.700, 0.668, 0.655), (7, 15)), ((0.700, 0.655, 0.668), (6, 15)),
                                     ((0.660, 0.655, 0.668), (6, 15)), ((0.660, 0.660, 0.660), (5, 15))])
def test_the_fastest_shape_wins(fmx, monkeypatch, ms, want):
    """The shape with the least time, by whatever margin; the first of equals."""
    from flashx_amd import tune
    import torch
    given = iter(ms)
    monkeypatch.setattr(tune, "_time_spmm", lambda spm, X, Y, reps: next(given))
    src, dst = fmx.rmat_edges(12, 16 << 12, 1)
    best, times, spm, _, _ = tune.autotune_tile(src, dst, 1 << 12, 4, torch.float32, keep=True)
    assert best == want and times == dict(zip(tune.DEFAULT_CANDIDATES, ms))
    assert spm.get_block_size() == (1 << want[0], 1 << want[1])
