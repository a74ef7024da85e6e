"""The tile that the float32 normalizer product takes at a size (host code, no GPU)."""
import ctypes

import pytest

from fast_rnnt_amd import _lib


def tile(B, S, T, C, windowed):
    waves = ctypes.c_int()
    return _lib.load().frnnt_simple_logprobs_tile(B, S, T, C, windowed, ctypes.byref(waves)), waves.value


# without windows every tile counts, and tall tiles are taken wherever they leave the fullest compute
# unit less to do: (B, S, T, C) -> (rows, waves)
@pytest.mark.parametrize("size,want", [
    ((1, 10, 50, 50), (32, 8)), ((16, 120, 400, 5000), (64, 8)), ((64, 40, 200, 1000), (64, 8)),
    ((32, 80, 250, 500), (96, 8)), ((32, 80, 250, 2500), (96, 8)), ((2, 240, 1256, 56), (32, 4)),
    ((23, 73, 202, 4093), (32, 8)), ((10, 137, 817, 500), (32, 4)), ((48, 90, 500, 250), (32, 4)),
    ((47, 53, 243, 1246), (32, 4)), ((70, 78, 565, 461), (32, 4)), ((2, 168, 1443, 79), (32, 4)),
    ((6, 137, 596, 134), (32, 4)),
    ((1, 0, 0, 1), (32, 8))])
def test_tiles_without_windows(size, want):
    assert tile(*size, 0) == want


@pytest.mark.parametrize("size,want", [
    ((1, 10, 50, 50), (32, 8)), ((16, 120, 400, 5000), (32, 8)), ((60, 50, 110, 2500), (64, 8)),
    ((32, 80, 250, 500), (96, 8)), ((30, 70, 250, 500), (32, 8)), ((64, 120, 600, 500), (32, 4))])
def test_tiles_with_windows(size, want):
    assert tile(*size, 1) == want


def test_bad_sizes_are_refused():
    assert _lib.load().frnnt_simple_logprobs_tile(0, 1, 1, 1, 0, None) == -1
    assert _lib.load().frnnt_simple_logprobs_tile(1, 1, 1, 0, 0, None) == -1
