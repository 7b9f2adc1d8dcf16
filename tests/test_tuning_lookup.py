"""tuning.lookup after the cache changed in place: a re-tuned entry (the same
key), a replaced one, and an exact batch before any other."""
from bpm_amd import tuning


def test_lookup_follows_the_cache(monkeypatch):
    cache = {"gfx950:64x64:1": {"best": [0, 1]}, "gfx950:64x64:16": {"best": [1, 6]},
             "gfx950:640x64:16": {"best": [2, 2]}, "gfx950:64x640:16": {"best": [2, 3]}}
    monkeypatch.setattr(tuning, "_cache", cache)
    assert tuning.lookup(64, 64, 1) == (0, 1) and tuning.lookup(64, 64, 40) == (1, 6)
    cache["gfx950:64x64:16"] = {"best": [5, 9]}     # re-tuned
    assert tuning.lookup(64, 64, 16) == (5, 9) and tuning.lookup(64, 64, 40) == (5, 9)
    cache["gfx950:64x64:1"]["best"] = [3, 4]
    assert tuning.lookup(64, 64, 1) == (3, 4)
    cache["gfx950:64x64:8"] = cache.pop("gfx950:64x64:1")   # as many entries, other keys
    assert tuning.lookup(64, 64, 1) == (3, 4) and tuning.lookup(64, 64, 8) == (3, 4)
    assert tuning.lookup(64, 128, 1) is None
