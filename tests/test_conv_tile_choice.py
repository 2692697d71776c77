"""Which tile a conv runs on, by the library's own kernel-name functions (no GPU): the lines at which the
tap classes change tiles, on both sides. The tiles themselves are held to float64 and to each other's
bits in test_gpu_conv_tiles.py."""
import ctypes
import re

import pytest

from dtts import lib
from dtts.nlc import ConvDesc

from test_gpu_conv_tiles import EPILOGUE, ROWS


def tile(lanes, length, cin, cout, k, dil=1):
    """(BM, BN, KC, stages, direct staging) of an f16 conv."""
    fn = getattr(lib(), "_ZN4dtts16conv_kernel_nameEPK14dtts_conv_desc")
    fn.restype = ctypes.c_char_p
    d = ConvDesc(lanes, length, cin, cout, k, dil, (k - 1) * dil)
    return _tile(fn(ctypes.byref(d)).decode())


def split_tile(lanes, length, cin, cout, k, dil=1):
    """The same of an f32 conv on the split route."""
    fn = getattr(lib(), "_ZN4dtts22conv_split_kernel_nameEllllll")
    fn.restype, fn.argtypes = ctypes.c_char_p, [ctypes.c_int64] * 6
    return _tile(fn(lanes, length, cin, cout, k, dil).decode())


def _tile(name):
    bm, bn, _, _, kc, _, _, stages, staging = map(int, re.search(r"ConvTile<([^>]*)>", name).group(1).split(", "))
    return bm, bn, kc, stages, staging == 1


@pytest.mark.parametrize("lanes,length,cin,cout,k,want", [
    # up to 159 register-staged workgroups of 256 x 64 (or 32): the small direct tiles
    (1, 3000, 256, 512, 7, (128, 64)), (1, 50, 256, 512, 3, (128, 32)), (159, 200, 64, 64, 7, (128, 64)),
    (159, 200, 64, 32, 5, (128, 32)),
    # from 160 on: register-staged
    (160, 200, 64, 64, 7, (256, 64)), (1, 6000, 256, 512, 7, (256, 64)), (48, 1500, 64, 160, 3, (256, 32)),
    (16, 3000, 256, 512, 7, (256, 64)), (48, 1500, 32, 32, 3, (256, 32)),
])
def test_narrow_widths_up_to_seven_taps(lanes, length, cin, cout, k, want):
    got = tile(lanes, length, cin, cout, k)
    assert got[:2] == want and got[4] == (want[0] == 128)


@pytest.mark.parametrize("lanes,length,channels,want", [
    (4, 16000, 192, (512, 96)), (1, 16000, 768, (512, 96)),  # one full round, or two of half the tile
    (24, 2000, 768, (512, 96)), (12, 10000, 384, (512, 96)), (4, 2000, 768, (256, 96)), (1, 1000, 384, (128, 32)),
    (1, 200, 768, (128, 32)), (8, 500, 384, (128, 64)),
])
def test_seven_taps(lanes, length, channels, want):
    assert tile(lanes, length, channels, channels, 7, 3)[:2] == want
    assert split_tile(lanes, length, channels, channels, 7, 3)[:2] == want


@pytest.mark.parametrize("lanes,length,cin,cout,want", [
    # 64 x 64 under the area of 192 tiles of 128 x 128 (128 at 96-multiples)
    (1, 25, 1536, 6144, (64, 64)), (191, 100, 384, 128, (64, 64)), (1, 9000, 768, 192, (64, 64)),
    (1, 9000, 384, 320, (64, 64)), (383, 128, 96, 64, (64, 64)), (85, 128, 96, 192, (64, 64)),
    # the large tiles from there on, register-staged where none divides the width
    (192, 100, 384, 128, (128, 128)), (4, 2000, 768, 1920, (256, 128)), (86, 128, 96, 192, (128, 96)),
    (1, 12000, 768, 192, (128, 96)), (384, 128, 96, 64, (256, 64)), (48, 5000, 512, 64, (256, 64)),
    (1, 12000, 384, 320, (256, 64)), (1, 100, 192, 288, (128, 96)),
])
def test_two_taps(lanes, length, cin, cout, want):
    assert tile(lanes, length, cin, cout, 2)[:2] == want
    if cout % 96 == 0 or cout % 128 == 0:  # widths the split route takes
        assert split_tile(lanes, length, cin, cout, 2)[:2] == want


@pytest.mark.parametrize("rows,cin,cout,want", [
    # few channels, many tiles: 32-channel stages, or 128 x 64
    (40000, 384, 384, (128, 128, 32)), (12000, 384, 384, (128, 64, 64)), (20000, 384, 384, (128, 128, 64)),
    (72000, 64, 64, (128, 64, 64)), (40000, 192, 192, (128, 64, 64)),
    # the estimate's five
    (701, 2048, 2048, (64, 64, 64)), (6400, 768, 768, (128, 64, 64)), (701, 2048, 12288, (256, 192, 64)),
    (2048, 2048, 4096, (128, 128, 64)), (2048, 6144, 2048, (128, 64, 64)), (3250, 1024, 4096, (256, 256, 64)), (129, 256, 2048, (64, 64, 64)),
])
def test_one_tap(rows, cin, cout, want):
    assert tile(1, rows, cin, cout, 1)[:3] == want
    assert tile(5, rows // 5, cin, cout, 1)[:3] == tile(1, rows // 5 * 5, cin, cout, 1)[:3]  # the lanes as one sequence


def _reached(rows):
    """Per tap class (7, 2, 1) the (BM, BN, KC) of the rows' convs, batched and one lane alone."""
    out = {7: set(), 2: set(), 1: set()}
    for lanes, length, cin, cout, k, dil in rows:
        for n in (lanes, 1):
            out[k if k <= 2 else 7].add(tile(n, length, cin, cout, k, dil)[:3])
    return out


def test_the_gpu_rows_reach_every_tile():
    got = _reached(ROWS)
    assert got[7] >= {(512, 96, 32), (256, 96, 32), (128, 96, 32), (128, 64, 32), (128, 32, 32), (256, 64, 32), (256, 32, 32)}
    assert got[2] >= {(256, 128, 32), (128, 128, 32), (128, 96, 32), (64, 64, 32), (256, 64, 32)}
    assert got[1] >= {(256, 256, 64), (256, 192, 64), (128, 128, 64), (128, 64, 64), (64, 64, 64), (128, 128, 32), (128, 96, 32)}
    got = _reached([(lanes, length, c, c, k, dil) for lanes, length, c, k, dil in EPILOGUE])
    assert got[7] >= {(512, 96, 32), (256, 96, 32), (128, 96, 32), (128, 64, 32), (128, 32, 32)}
    assert got[1] >= {(256, 256, 64), (128, 128, 64), (128, 64, 64), (64, 64, 64), (128, 128, 32)}
