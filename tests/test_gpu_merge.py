"""merge_sorted (multiset union) around the edges of its merge-path tiles of
8192 values: lists of every size ratio, empty and disjoint ones, equal values
within and across tiles, and more copies on either side."""
import numpy as np
import pytest

import engine_amd as ea
from engine_amd import datagen
from engine_amd.formats import uncompr_f

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ea.init(0)


def union(a, b):
    """Each value as often as in the list that has more of it."""
    v = np.union1d(a, b)
    count = lambda x: np.searchsorted(x, v, side="right") - np.searchsorted(x, v, side="left")  # noqa: E731
    return np.repeat(v, np.maximum(count(a), count(b)))


@pytest.mark.parametrize("na,nb", [(0, 0), (0, 5), (5, 0), (1, 1), (4096, 4096), (4096, 4097), (8191, 1), (1, 8192),
                                   (8193, 8193), (100_000, 3), (3, 100_000), (50_000, 70_000), (300_000, 290_000)])
@pytest.mark.parametrize("bits", [2, 6, 16, 40])
def test_merge(na, nb, bits):
    a = np.sort(datagen.uniform_bits(7 + na, na, bits))
    b = np.sort(datagen.uniform_bits(1000 + nb, nb, bits))
    got = ea.merge_sorted(uncompr_f(), ea.upload_values(a), ea.upload_values(b)).values()
    assert np.array_equal(got, union(a, b))


@pytest.mark.parametrize("na,nb", [(20_000, 20_000), (20_000, 9_000), (9_000, 20_000)])
def test_merge_one_value_and_disjoint(na, nb):
    for a, b in [(np.full(na, 5), np.full(nb, 5)), (np.arange(na), np.arange(nb) + na),
                 (np.arange(na) + nb, np.arange(nb)), (np.arange(na), np.arange(nb)),
                 (np.full(na, 2**64 - 1), np.full(nb, 2**64 - 1))]:
        a, b = a.astype(np.uint64), b.astype(np.uint64)
        got = ea.merge_sorted(uncompr_f(), ea.upload_values(a), ea.upload_values(b)).values()
        assert np.array_equal(got, union(a, b))


def test_merge_many_tiles():
    # 4800 tiles, several per resident workgroup: its staged values are reused
    r = datagen.splitmix64(3, 2 * 20_000_000)
    gaps = (r >> np.uint64(62)) + np.uint64(1)
    a, b = np.cumsum(gaps[:20_000_000], dtype=np.uint64), np.cumsum(gaps[20_000_000:], dtype=np.uint64)
    either = np.zeros(int(max(a[-1], b[-1])) + 1, bool)
    either[a] = either[b] = True
    got = ea.merge_sorted(uncompr_f(), ea.upload_values(a), ea.upload_values(b)).values()
    assert np.array_equal(got, np.flatnonzero(either).astype(np.uint64))
