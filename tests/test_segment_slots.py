"""The segments' buffer (jax-gs_amd/csrc/gs_segments.h): the slots that tiles get, for any lists, and
its size, which is what every live render holds until its backward."""
import os
import subprocess

import pytest

from jax_gs_amd import _lib
from test_cull import _CSRC, HIPCC

_HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def slots_bin(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    out = str(tmp_path_factory.mktemp("segments") / "segment_slots")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-I", _CSRC, os.path.join(_HERE, "segment_slots.cpp"), "-o", out],
                   check=True, capture_output=True)
    return out


@pytest.mark.parametrize("seed", [1, 2])
def test_tiles_slots_are_their_own(slots_bin, seed):
    res = subprocess.run([slots_bin, "3000", str(seed)], capture_output=True, text=True)
    sets, packed, faults = (int(v) for v in res.stdout.split())
    assert faults == 0 and res.returncode == 0
    assert sets // 5 < packed < sets - sets // 20  # both kinds of layout


@pytest.mark.parametrize("w,h", [(504, 378), (640, 479), (979, 546), (1440, 1079)])
def test_held_bytes_follow_the_capacity(w, h):
    """4 KB per segment: one per tile and one per 64 (below 2048 tiles) or 128 entries, and never
    more than lists of any length take."""
    L = _lib.lib()
    T = ((w + 15) // 16) * ((h + 15) // 16)
    unit, most = (64, 32) if T < 2048 else (128, 16)
    full = L.gs_composite_segments_size(w, h)
    side = 4 * (2 + 4 * T + 2048) + 4 * T * 16 + 1024  # work items and counts
    assert 4096 * T * most <= full <= 4096 * T * most + side
    for cap in (1, 1000, T * 8, T * 300, 256 * 2000):
        size = L.gs_composite_segments_size_for(w, h, cap)
        assert size <= min(full, 4096 * (T + cap // unit) + side)
    assert L.gs_composite_segments_size_for(w, h, 2 ** 31 - 1) == full
    # from 6144 tiles on: the order of the tiles
    assert L.gs_composite_segments_size_for(1920, 1080, 1000) == L.gs_composite_segments_size(1920, 1080) == 4 * 8160
