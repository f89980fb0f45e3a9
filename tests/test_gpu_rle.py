"""rle_f compression and expansion around the edges of their units (rows of
128 values, waves of 2048, tiles of 16384, 256 heads of a wave kept in LDS;
output windows of 4096 values): images equal the oracle's and the round trip
is exact."""
import numpy as np
import pytest

import engine_amd as ea
from engine_amd import datagen
from engine_amd.formats import rle_f, uncompr_f

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 127, 129, 2047, 2048, 4097, 16384, 16385, 3 * 16384 + 2049, 70 * 16384 + 77]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ea.init(0)


def runs_of(lens, n):
    """Runs of the given lengths, repeated up to n values; neighbours differ."""
    lens = np.resize(np.asarray(lens, dtype=np.int64), n)
    k = int(np.searchsorted(np.cumsum(lens), n)) + 1
    v = datagen.splitmix64(77, k) * np.uint64(2) + (np.arange(k, dtype=np.uint64) & np.uint64(1))
    return np.repeat(v, lens[:k])[:n]


@pytest.mark.parametrize("lens", [[1], [2], [7], [8], [9], [64], [2048], [16384], [1 << 40], [1, 5000, 3, 1, 1, 90],
                                  [2047, 1], [16383, 2, 16383], [1] * 2000 + [100000]], ids=lambda x: str(x[:4]))
def test_rle_both_ways(oracle, lens):
    for n in SIZES:
        v = runs_of(np.minimum(lens, n), n)
        g = ea.morph(rle_f(), ea.upload_values(v))
        o = oracle.morph(rle_f(), v)
        img, meta = g.image()
        assert meta == o.meta(), n
        assert img.tobytes() == o.image().tobytes(), n
        assert np.array_equal(ea.morph(uncompr_f(), g).values(), v), n


@pytest.mark.parametrize("lens", [[1, 2], [5] * 20_000 + [9] * 20_000], ids=lambda x: str(x[:2]))
def test_rle_both_ways_many_tiles(oracle, lens):
    # 4096 tiles, several per resident workgroup: its kept heads are reused;
    # every wave beyond its 256 kept heads, and waves on either side of that
    v = runs_of(lens, 1 << 26)
    g = ea.morph(rle_f(), ea.upload_values(v))
    o = oracle.morph(rle_f(), v)
    img, meta = g.image()
    assert meta == o.meta() and np.array_equal(img, o.image())
    assert np.array_equal(ea.morph(uncompr_f(), g).values(), v)
