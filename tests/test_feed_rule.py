"""How traversal launches deal rays to their waves (kp_feed.h, compiled alone
with the host compiler): for any grid, also ones that do not hold five waves a
SIMD (the 4-wave builds, a scratch or a tuning that allows fewer blocks), every
ray is in exactly one first chunk or left to the work counter, the counter is
used exactly when the launch clears it, and a thin launch uses one wave per
SIMD, or two, of the SIMDs that the grid reaches."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "kp_feed.h"
extern "C" {
uint32_t first_chunk(uint32_t n, uint32_t waves, uint32_t simds, uint32_t one, uint32_t most, int even) {
    return kp::first_chunk(n, waves, simds, one, most, even != 0);
}
int hold_all(uint32_t n, uint32_t waves) { return kp::first_chunks_hold_all(n, waves); }
uint32_t limit(int any, int most) {
    return any ? (most ? kp::kThinMost<true> : kp::kThinOne<true>) : (most ? kp::kThinMost<false> : kp::kThinOne<false>);
}
uint32_t chunk() { return kp::kChunk; }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("feed")
    (d / "feed.cpp").write_text(SRC)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                        "-I" + os.path.join(ROOT, "kazen_proto_amd", "csrc"), str(d / "feed.cpp"), "-o",
                        str(d / "feed.so")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return ctypes.CDLL(str(d / "feed.so"))


# blocks of four waves, SIMDs of the device
GRIDS = [(1280, 1024), (1024, 1024), (256, 1024), (205, 1024), (96, 1024), (1, 1024), (2, 1024), (512, 1024),
         (1280, 1216), (3, 4), (1, 4)]


def _counts(waves, simds):
    base = {1, 2, 3, 63, 64, 65}
    for k in (1, 8, 32, 64, 128, 256):
        for w in (waves, min(waves, simds), 2 * min(waves, simds)):
            base |= {k * w - 1, k * w, k * w + 1}
    base |= {waves * 511, waves * 512 + 1, waves * 9000 + 7, 1 << 26, (1 << 32) - 1}
    return sorted(n for n in base if 0 < n < 1 << 32)


@pytest.mark.parametrize("blocks,simds", GRIDS)
@pytest.mark.parametrize("any_hit", [0, 1])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("even", [0, 1])
def test_first_chunks(rule, blocks, simds, any_hit, split, even):
    waves = 4 * blocks
    one, most = rule.limit(any_hit, 0), rule.limit(any_hit, 1) if split else 0
    reached = min(waves, simds)
    for n in _counts(waves, simds):
        f = rule.first_chunk(n, waves, simds, one, most, even)
        assert f > 0 and f * waves < 1 << 32
        assert bool(rule.hold_all(n, waves)) == (n <= waves * rule.chunk())
        if rule.hold_all(n, waves):          # the counter is not cleared, so it must not be needed
            assert f * waves >= n
        used = -(-n // f)
        if split and n <= reached * most:
            want = reached if n <= reached * one else min(waves, 2 * reached)
            assert f == -(-n // want) and used <= want
        elif not even:
            assert f % 64 == 0
    assert rule.first_chunk(0, waves, simds, one, most, even) * waves >= 0


def test_a_four_wave_grid_spreads_over_every_simd(rule):
    """1,000 closest-hit rays on 256 CUs: a ray per wave, whether the grid
    holds four or five waves a SIMD."""
    for blocks in (1024, 1280, 256):
        assert rule.first_chunk(1000, 4 * blocks, 1024, rule.limit(0, 0), rule.limit(0, 1), 0) == 1
        assert rule.first_chunk(8192, 4 * blocks, 1024, rule.limit(0, 0), rule.limit(0, 1), 0) == 8
