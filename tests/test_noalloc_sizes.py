"""Sizes of the allocation-free entry point: the bytes it reports are those its
kernels use, and the sizes it takes are those whose buffers fit 64 MiB beside
the distance field's last band of rows.  Needs no GPU."""
import ctypes

import pytest

import radiancecascade_amd as rc
from radiancecascade_amd import _abi


def _up(x, m):
    return -(-x // m) * m


def _need(W, H, L, rows):
    bands = -(-H // 64)
    total = _up(8 * bands * W, 256) + _up(4 * bands * W, 256) + _up(_up(W, 16) * rows, 256)
    for i in range(1, L):
        px, py = rc.probe_grid(W, H, i)
        total += _up(px * py * 4 ** i * 16, 256)
    return total


@pytest.mark.parametrize("W,H,L", [(1, 1, 1), (64, 64, 3), (17, 8, 2), (1920, 1080, 6), (1283, 717, 6), (16384, 16384, 1),
                                   (16380, 256, 1), (255, 16384, 7)])
def test_reported_bytes_hold_the_field_with_its_row_of_zeros(W, H, L):
    """A row of zeros lies below the image's last: 8 rows more where the height
    is a multiple of 8."""
    assert _abi.load().rc_noalloc_scratch_bytes(W, H, L) == _need(W, H, L, _up(H + 1, 8))


@pytest.mark.parametrize("W,L", [(2048, 7), (2000, 6), (1111, 3), (16384, 2), (16370, 1), (333, 1), (3000, 1), (4104, 1)])
def test_sizes_taken_are_those_without_the_last_band(W, L):
    if rc.device_count() > 0:
        pytest.skip("a size that is taken would run")
    lib = _abi.load()
    g = _abi.GBuffer(256, 0, 256)

    def taken(H):
        return lib.rc_run_device_noalloc(W, H, L, ctypes.byref(g), 256, None) != _abi.ERR_INVALID

    lo, hi = 0, 16384
    while lo < hi:
        mid = (lo + hi + 1) // 2
        lo, hi = (mid, hi) if _need(W, mid, L, _up(mid, 8)) <= 64 << 20 else (lo, mid - 1)
    for H in {1, 8, *range(max(1, lo - 70), min(16384, lo + 70) + 1)}:
        assert taken(H) == (_need(W, H, L, _up(H, 8)) <= 64 << 20), H
