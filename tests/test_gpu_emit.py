"""The single-pass emission of 8-lane 512-value blocks: byte images equal
the oracle's around the edges of its units (blocks, waves of 4 blocks,
tiles of 32, pages of 64 and 2048), for every cascade depth it takes and
those it leaves to the general path, and for blocks of any width (more than
32 bits take another way through it)."""
import numpy as np
import pytest

import engine_amd as ea
from engine_amd import datagen
from engine_amd.formats import MS_OP_XOR, delta_f, dynamic_vbp_f, for_f

pytestmark = pytest.mark.gpu

INNER = dynamic_vbp_f(512, 64, 8)
FORMATS = [dynamic_vbp_f(512, 64, 8), dynamic_vbp_f(512, 2048, 8), dynamic_vbp_f(512, 192, 8),
           delta_f(512, 8, INNER), delta_f(1024, 8, INNER), delta_f(2048, 8, INNER), delta_f(4096, 8, INNER),
           for_f(512, 8, INNER), for_f(1024, 8, INNER), for_f(2048, 8, INNER), for_f(1024, 32, INNER)]
SIZES = [511, 512, 2047, 2048 + 512, 16384 - 512, 16384, 16384 + 1, 5 * 16384 + 2048 + 333, 2049 * 512 + 5]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ea.init(0)


def values(kind, n):
    r = datagen.splitmix64(0x4D6F7270 + n, n)
    if kind == "narrow":         # widths 1..32, one per block
        return r >> np.uint64(32) >> (np.arange(n, dtype=np.uint64) // 512 * 7 % 32)
    if kind == "wide":           # every width up to 64, alone in a wave of narrow blocks and together
        return r >> (np.arange(n, dtype=np.uint64) // 512 * 11 % 64)
    if kind == "zero":
        return np.zeros(n, np.uint64)
    return np.cumsum(r >> np.uint64(59), dtype=np.uint64) + np.uint64(1 << 50)   # sorted


def same(g, o):
    img, meta = g.image()
    assert meta == o.meta()
    assert img.tobytes() == o.image().tobytes()


@pytest.mark.parametrize("f", FORMATS, ids=repr)
@pytest.mark.parametrize("kind", ["narrow", "wide", "zero", "sorted"])
def test_column_emission(oracle, f, kind):
    for n in SIZES:
        v = values(kind, n)
        same(ea.morph(f, ea.upload_values(v)), oracle.morph(f, v))


@pytest.mark.parametrize("f", FORMATS[:6] + FORMATS[7:10], ids=repr)
def test_write_iterator_emission(oracle, f):
    # x xor 0 through the write-iterator: calls of 2048 values, fresh pages each
    for n in SIZES:
        v, z = values("wide", n), np.zeros(n, np.uint64)
        g = ea.calc_binary(MS_OP_XOR, f, ea.upload_values(v), ea.upload_values(z))
        o = oracle.calc_binary(MS_OP_XOR, f, oracle.morph(ea.FormatDesc(0), v), oracle.morph(ea.FormatDesc(0), z))
        same(g, o)


@pytest.mark.parametrize("f", [FORMATS[0], FORMATS[4], FORMATS[8]], ids=repr)
def test_column_emission_many_tiles(oracle, f):
    # 4096 tiles, several per resident workgroup: its words, references and
    # deferred tile are reused; blocks of every width, so that tiles packed in
    # LDS and tiles with blocks read again follow each other
    v = values("wide", 1 << 26)
    same(ea.morph(f, ea.upload_values(v)), oracle.morph(f, v))
