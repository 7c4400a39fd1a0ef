"""How the gather kernels' waves are dealt the windows of a graph (csrc/schedule.hpp, compiled here for the host): every tile once, parts that cover
their window, waves of like length.  No GPU needed."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hopper_spmm_amd", "csrc")
SOURCE = """
#include "schedule.hpp"
using namespace hspmm;
static Schedule s;
extern "C" unsigned make(unsigned W, const uint32_t *rowOffset, unsigned waves) { s = build_schedule(W, rowOffset, waves); return unsigned(s.items.size()); }
extern "C" const uint32_t *items() { return &s.items[0].window; }
extern "C" const uint32_t *waves() { return s.waves.data(); }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    at = tmp_path_factory.mktemp("schedule")
    (at / "schedule.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, "-o", str(at / "schedule.so"), str(at / "schedule.cpp")], check=True)
    lib = ctypes.CDLL(str(at / "schedule.so"))
    lib.items.restype = lib.waves.restype = ctypes.POINTER(ctypes.c_uint32)
    return lib


@pytest.mark.parametrize("tiles,n_waves", [([1], 1), ([1], 4), ([100], 64), ([5, 5, 5], 2), ([1] * 1000, 16), ([3000] + [2] * 500, 64), (None, 7), (None, 256)])
def test_every_tile_once_and_waves_alike(host, tiles, n_waves):
    tiles = np.array(tiles if tiles is not None else np.random.default_rng(n_waves).zipf(1.7, 5000).clip(1, 2000))
    offset = np.concatenate([[0], np.cumsum(tiles)]).astype(np.uint32)
    n = host.make(len(tiles), offset.ctypes.data_as(ctypes.c_void_p), n_waves)
    items = np.ctypeslib.as_array(host.items(), (n, 6)).astype(np.int64)
    waves = np.ctypeslib.as_array(host.waves(), (n_waves + 1,)).astype(np.int64)
    seen = np.concatenate([first + stride * np.arange(steps) for _, first, stride, steps, _, _ in items])
    assert (np.sort(seen) == np.arange(offset[-1])).all()
    window, first, stride, steps, part, parts = items.T
    assert (steps >= 1).all() and (stride == parts).all() and (first == offset[window] + part).all() and (first + stride * (steps - 1) < offset[window + 1]).all()
    share = -(-int(offset[-1]) // n_waves)
    assert (parts == -(-tiles[window] // share)).all() and (steps <= share).all()
    assert waves[0] == 0 and waves[-1] == n and (np.diff(waves) >= 0).all()
    # the first waves are the ones that have items, and the longest item is the most that two of them differ by
    assert (np.diff(waves)[:min(n, n_waves)] > 0).all()
    cost = np.array([(2 * steps[a:b] + 3).sum() for a, b in zip(waves[:-1], waves[1:])])
    assert cost.max() - cost.min() <= 2 * steps.max() + 3
    assert all((np.diff(steps[a:b]) <= 0).all() for a, b in zip(waves[:-1], waves[1:]))
