"""CPU: which attention kernels a launch takes (soupk_attention_wide: 128 or 64 queries per workgroup)
against what both measured on MI355X (256 CUs, graph replays, best of the runs): the faster one
wherever the two differ by more than 4%, apart from the cases listed as left to the other."""

import ctypes

import pytest

from testt_amd import _ext

CUS = 256
LEVEL = 0.04


def wide(varlen, backward, B, length, NH, cus=CUS):
    out = ctypes.c_int32(-1)
    _ext.call("soupk_attention_wide", varlen, backward, B, length, NH, cus, ctypes.addressof(out))
    return bool(out.value)


def check(takes_wide, narrow_us, wide_us):
    if abs(narrow_us - wide_us) > LEVEL * min(narrow_us, wide_us):
        assert takes_wide == (wide_us < narrow_us)


def ragged(seq, rows):
    return [seq // (i + 1) for i in range(rows)]


# (rows, positions, heads, 64-query us, 128-query us)
PADDED_FWD = [(43, 32, 12, 12.4, 13.0), (28, 64, 12, 11.2, 11.1), (43, 64, 12, 15.4, 16.4),
              (80, 64, 12, 22.8, 21.5), (28, 96, 12, 16.6, 14.9), (80, 96, 12, 41.1, 30.2),
              (28, 128, 12, 17.6, 17.1), (80, 128, 12, 43.7, 35.1), (14, 160, 12, 14.3, 15.8),
              (22, 160, 12, 22.7, 24.4), (40, 160, 12, 35.4, 31.0), (14, 192, 12, 15.0, 16.2),
              (22, 192, 12, 24.3, 26.8), (40, 192, 12, 37.1, 32.9), (6, 160, 28, 14.1, 15.6),
              (10, 192, 28, 24.8, 26.9), (14, 256, 12, 20.9, 19.4), (40, 256, 12, 51.8, 38.2),
              (8, 512, 12, 32.1, 28.8), (4, 1024, 12, 51.5, 46.9), (2, 2048, 12, 88.1, 81.5)]
PADDED_BWD = [(28, 16, 12, 18.4, 21.7), (128, 32, 12, 54.3, 65.0), (64, 64, 12, 50.5, 54.4),
              (32, 100, 12, 46.3, 49.4), (43, 128, 12, 66.3, 72.3), (14, 160, 12, 38.3, 44.6),
              (16, 200, 12, 53.6, 57.6), (40, 192, 12, 95.0, 105.8), (14, 256, 12, 56.3, 55.0),
              (40, 256, 12, 131.0, 134.0), (4, 320, 28, 50.2, 54.8), (10, 320, 12, 53.6, 56.4),
              (10, 384, 12, 66.1, 64.5), (7, 512, 12, 70.9, 66.3), (20, 512, 12, 177.0, 162.0),
              (8, 768, 12, 134.0, 122.0), (4, 1024, 12, 108.4, 98.1), (3, 1536, 12, 162.0, 141.0)]


@pytest.mark.parametrize("B,T,NH,narrow_us,wide_us", PADDED_FWD)
def test_padded_forward(B, T, NH, narrow_us, wide_us):
    check(wide(0, 0, B, T, NH), narrow_us, wide_us)


@pytest.mark.parametrize("B,T,NH,narrow_us,wide_us", PADDED_BWD)
def test_padded_backward(B, T, NH, narrow_us, wide_us):
    check(wide(0, 1, B, T, NH), narrow_us, wide_us)


# (row lengths, heads, 64-query us, 128-query us)
VARLEN_FWD = [([64] * 27, 12, 16.8, 10.6), ([64] * 64, 12, 60.9, 28.1), ([65] * 20, 28, 31.0, 19.4),
              ([129] * 16, 12, 19.4, 14.7), ([256] * 16, 12, 32.5, 20.2), ([700] * 5, 12, 31.5, 27.1),
              ([1024] * 4, 12, 40.6, 34.0), ([1300] * 3, 12, 48.3, 41.4), ([4096], 12, 119.9, 107.1),
              ([4096] * 2, 12, 222.0, 141.0), ([512] * 4, 12, 15.4, 20.5), ([3000], 12, 75.0, 82.0),
              ([1365] * 2, 12, 36.0, 42.0), ([4096] + [16] * 31, 12, 306.7, 160.8),
              (ragged(1696, 3), 12, 45.7, 51.4), (ragged(1504, 4), 12, 39.8, 45.1),
              (ragged(2592, 2), 12, 80.6, 71.9), (ragged(1984, 4), 12, 63.7, 55.7),
              (ragged(1536, 8), 12, 64.2, 47.2), (ragged(640, 16), 12, 24.6, 23.9),
              ([1120] + [140] * 7, 14, 28.2, 35.5), (ragged(768, 8), 14, 21.1, 26.2),
              (ragged(512, 4), 28, 18.9, 20.9), (ragged(640, 3), 28, 21.6, 25.3),
              (ragged(1280, 3), 16, 31.8, 38.3), ([2304, 288], 14, 67.7, 67.5)]
VARLEN_BWD = [([64] * 27, 12, 43.3, 39.4), ([64] * 64, 12, 151.0, 130.0), ([128] * 32, 12, 101.7, 88.5),
              ([256] * 16, 12, 84.5, 73.1), ([1000] * 4, 12, 98.5, 92.5), ([4096], 12, 275.7, 240.5),
              ([3500], 12, 208.1, 188.3), (ragged(1696, 3), 12, 97.8, 96.5),
              (ragged(1504, 4), 12, 94.1, 88.6), (ragged(640, 16), 12, 56.8, 52.5),
              (ragged(512, 4), 28, 46.1, 48.5), (ragged(384, 8), 28, 43.6, 46.0),
              (ragged(256, 4), 40, 34.7, 37.4), (ragged(448, 3), 40, 47.9, 51.2),
              ([64] + [8] * 7, 40, 18.2, 19.6), ([512] * 4, 12, 40.0, 42.0)]
# where the rule takes the slower kernel: the row lengths, which lie on the device, decide there
LEFT_FWD = [(ragged(1888, 3), 12, 50.7, 55.7), ([3104, 388, 388], 12, 88.1, 96.3),
            ([513] * 6, 12, 28.6, 23.7), ([2080, 260], 16, 88.0, 58.1)]


@pytest.mark.parametrize("lengths,NH,narrow_us,wide_us", VARLEN_FWD)
def test_varlen_forward(lengths, NH, narrow_us, wide_us):
    check(wide(1, 0, len(lengths), sum(lengths), NH), narrow_us, wide_us)


@pytest.mark.parametrize("lengths,NH,narrow_us,wide_us", VARLEN_BWD)
def test_varlen_backward(lengths, NH, narrow_us, wide_us):
    check(wide(1, 1, len(lengths), sum(lengths), NH), narrow_us, wide_us)


@pytest.mark.parametrize("lengths,NH,narrow_us,wide_us", LEFT_FWD)
def test_varlen_forward_left(lengths, NH, narrow_us, wide_us):
    assert wide(1, 0, len(lengths), sum(lengths), NH) != (wide_us < narrow_us)


def test_empty_and_invalid():
    assert not wide(1, 0, 0, 0, 12) and not wide(0, 1, 0, 512, 12) and not wide(0, 0, 4, 0, 12)
    assert not wide(1, 1, 4, 0, 12)
    for bad in ((0, 0, -1, 64, 12), (0, 0, 1, -1, 12), (0, 0, 1, 64, 0), (0, 0, 1, 64, 12, 0)):
        with pytest.raises(_ext.SoupkError):
            wide(*bad)
