"""The autotuner times only candidates that launch different things."""
from apogee_amd import autotune


def test_flat_tiles_that_the_filter_keeps():
    # four transforms of 1024 points share a workgroup: 256 groups of templates
    assert autotune.flat_tiles(1024, 16, 1024) == [1, 2, 4]
    assert autotune.flat_tiles(4096, 16, 1024) == [1, 2, 4, 8, 16]
    assert autotune.flat_tiles(4096, 4, 4096) == [1, 2, 4]
    assert autotune.flat_tiles(4096, 64, 256) == [1, 2, 4, 8, 16]
    assert autotune.flat_tiles(4096, 2, 512) == [1]
    assert autotune.flat_tiles(16384, 16, 256) == [1]
    assert autotune.flat_tiles(65536, 4, 128) == [1]


class _Timed:
    """Stands for a device context: records the tuning keys it is given."""

    def __init__(self, *args):
        self.keys = []

    def set_tuning(self, key, value):
        self.keys.append((key, value))

    def __getattr__(self, name):
        return lambda *a, **k: None


def test_chunk_sizes_are_timed_on_the_path_that_has_chunks(monkeypatch):
    import numpy as np
    import torch
    from apogee_amd import _hip
    made = []
    monkeypatch.setattr(_hip, "Context", lambda *a: made.append(_Timed()) or made[-1])
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: empty(1))
    monkeypatch.setattr(autotune, "_median_ms", lambda *a: 1.0)
    autotune._tune_big(0, 32768, 1, 1, 1024, 1, np.random.default_rng(0))
    keys = made[0].keys
    assert keys[0] == ("wide", 2) and ("big_chunk_mb", 64) in keys
    autotune._tune_flat(0, 16384, 1, 1, 16384, 1, np.random.default_rng(0))
    assert made[1].keys == [("dpw", 1)]
