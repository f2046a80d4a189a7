"""Strided gathers against NumPy strides, bit for bit: transposes at the edges
of the 64 x 64 tiles and at the shortest axes that use them, row copies whose
vector runs cross row ends, strided, reversed and repeated (stride 0) axes, in
every word size; and the same routes under offsets that leave the source
aligned to one element only."""

import numpy as np
import pytest

import openpacho as p

pytestmark = pytest.mark.gpu

# (source elements, offset, shape, strides): every index lies in the source.
FORMS = {
    "square": (130 * 130, 0, (130, 130), (1, 130)),
    "tile": (64 * 64, 0, (64, 64), (1, 64)),
    "tile+1": (65 * 63, 0, (65, 63), (1, 65)),
    "shortest": (16 * 40 + 3, 3, (16, 40), (1, 16)),
    "below": (15 * 300, 0, (15, 300), (1, 15)),
    "thin": (3 * 5000, 0, (3, 5000), (1, 3)),
    "batched": (5 * 70 * 33, 0, (5, 33, 70), (70 * 33, 1, 33)),
    "outer-lane": (40 * 9 * 50, 0, (40, 9, 50), (1, 40, 360)),
    "lane-step": (80 * 200 + 7, 7, (40, 200), (2, 80)),
    "lane-back": (70 * 100, 69, (70, 100), (-1, 70)),
    "rows-back": (70 * 100, 99 * 70, (70, 100), (1, -70)),
    "rows": (50 * 131 + 1, 1, (50, 130), (131, 1)),
    "short-rows": (999 * 5, 2, (999, 3), (5, 1)),
    "stretch": (100001, 1, (100000,), (1,)),
    "every-other": (40 * 501, 1, (40, 250), (501, 2)),
    "reversed": (1000, 999, (1000,), (-1,)),
    "repeated": (77, 0, (90, 77), (0, 1)),
    "repeated-inner": (77, 0, (77, 90), (1, 0)),
    "rank8": (2**8, 0, (2,) * 8, tuple(2 ** (7 - (3 * d) % 8) for d in range(8))),
    "one": (9, 8, (), ()),
    # Either side of the shares of a tile that decide for or against tiles.
    "third": (32 * 43, 0, (32, 43), (1, 32)),
    "below a third": (32 * 42, 0, (32, 42), (1, 32)),
    "quarter": (16 * 256, 0, (16, 256), (1, 16)),
    "below a quarter": (3 * 14 * 250, 0, (3, 14, 250), (14 * 250, 1, 14)),
    "fifth": (12 * 1152, 0, (12, 1152), (1, 12)),
    "below a fifth": (11 * 1100, 0, (11, 1100), (1, 11)),
    "sliver": (5 * 100 * 65, 0, (5, 100, 65), (6500, 1, 100)),
    "wide sliver": (5 * 128 * 65, 0, (5, 128, 65), (8320, 1, 128)),
}


@pytest.mark.parametrize("dtype", [np.bool_, np.float32, np.int64])
@pytest.mark.parametrize("name", FORMS)
def test_gathers_match_numpy_strides(hip, name, dtype):
    size, offset, shape, strides = FORMS[name]
    bits = np.random.default_rng(len(name)).integers(0, 256, size * np.dtype(dtype).itemsize, dtype=np.uint8)
    host = (bits & 1).astype(np.bool_) if dtype == np.bool_ else bits.view(dtype)
    raw = host.view(f"u{host.itemsize}")  # NaN payloads compare as words
    want = np.lib.stride_tricks.as_strided(raw[offset:], shape, [s * raw.itemsize for s in strides])
    source = p.asarray(host, backend=hip)
    got = p.ndarray._wrap(hip.gather(source, shape, offset, strides), shape, host.dtype, hip)
    np.testing.assert_array_equal(p.asnumpy(got).view(raw.dtype), want)


# (elements, row): the last workgroup's overhang (2048 elements) passes 31 bits
# from 2^31 - 2047 elements on: 64-bit indices there, 32-bit ones before.
@pytest.mark.parametrize("count,length", [(2**31 - 2048, 384), (2**31 - 2046, 14), (2**31 - 2, 331)])
def test_gathers_at_the_largest_arrays(hip, count, length):
    host = np.random.default_rng(count).integers(0, 2, length).astype(np.bool_)
    source = p.asarray(host, backend=hip)
    shape = (count // length, length)  # one row, read again and again
    got = p.asnumpy(p.ndarray._wrap(hip.gather(source, shape, 0, (0, 1)), shape, host.dtype, hip))
    for rows in np.array_split(got, 64):
        assert np.array_equal(rows, np.broadcast_to(host, rows.shape))
