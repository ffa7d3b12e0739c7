"""The search for a batch's configuration (kazan_tune: the tuner over given
times): what it tries, that it never tries what does not build, and that the
runs that decide are of different configurations."""
import ctypes
import itertools

import numpy as np
import pytest

MS = ctypes.CFUNCTYPE(ctypes.c_float, ctypes.POINTER(ctypes.c_uint32))
ALL = [c for c in itertools.product((8, 16, 32, 64), (1, 2, 4), (0, 1), (0, 1), (0, 1, 2), (1, 4, 16))]


def _tune(driver, times, own=16, largest=64, model=1):
    """times: {configuration: ms}; returns (trials, choice)."""
    seen = []

    def ms(p):
        c = tuple(p[:6])
        seen.append(c)
        return times[c]

    fn = MS(ms)
    trials, choice = (ctypes.c_uint32 * (6 * 64))(), (ctypes.c_uint32 * 6)()
    n = driver.lib.kazan_tune(own, largest, model, fn, trials, 64, choice)
    assert n == len(seen)
    assert [tuple(trials[6 * i:6 * i + 6]) for i in range(n)] == seen
    return seen, tuple(choice)


def _random_times(seed, favour=None):
    r = np.random.default_rng(seed)
    t = dict(zip(ALL, r.uniform(1.0, 2.0, len(ALL))))
    if favour:
        t = {c: (v - 0.9 if favour(c) else v) for c, v in t.items()}
    return t


@pytest.mark.parametrize("seed", range(20))
@pytest.mark.parametrize("favour", [None, lambda c: c[3] == 0, lambda c: c[3] == 1, lambda c: c[5] == 16])
def test_finalists_differ(driver, seed, favour):
    times = _random_times(seed, favour)
    for model in (0, 1):
        trials, choice = _tune(driver, times, model=model)
        finals = trials[-6:]
        assert finals[0] == finals[1] and finals[2] == finals[3] and finals[4] == finals[5]
        assert len({finals[0], finals[2], finals[4]}) == 3, finals
        # noise-free times: the three fastest of all that was tried, the fastest kept
        assert [finals[0], finals[2], finals[4]] == sorted(set(trials[:-6]), key=times.get)[:3]
        assert choice == min(trials, key=times.get)


@pytest.mark.parametrize("own", [8, 16, 32])
def test_own_tile_size_last_of_the_sizes(driver, own):
    trials, _ = _tune(driver, _random_times(1), own=own)
    assert [c[0] for c in trials[:4]] == [s for s in (8, 16, 32, 64) if s != own] + [own]


@pytest.mark.parametrize("largest", [16, 32, 64])
@pytest.mark.parametrize("tile", [8, 16, 32, 64])
def test_only_what_builds_is_tried(driver, largest, tile):
    """Whatever tile size is the fastest, planned and plain (the plain raster's larger neighbour included)."""
    if tile > largest:
        pytest.skip("does not fit")
    for plain in (False, True):
        times = {c: (1.0 if c[0] == tile else 2.0) + (0.5 if (c[3] == 0) != plain else 0.0) for c in ALL}
        trials, choice = _tune(driver, times, largest=largest)
        assert all(c[0] <= largest for c in trials)
        assert choice[0] == tile and choice[3] == (0 if plain else 1)
