"""Positions of a select into uncompr_f in one pass: every source layout (8
lanes, one lane, raw values, others decompressed first) at the edges of its
units (512 rows), blocks (64 rows of one lane) and tiles, for selections
from none to all of the rows and each number of units per wave."""
import numpy as np
import pytest

import engine_amd as ea
from engine_amd import datagen
from engine_amd.formats import (MS_CMP_EQ, MS_CMP_GE, MS_CMP_LT, MS_CMP_NE, default_delta_dynamic_vbp_f,
                                default_for_dynamic_vbp_f, dynamic_vbp_f, rle_f, static_vbp_f, uncompr_f)
from tests import refmodel as rm

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 63, 64, 65, 511, 513, 575, 8192 - 1, 8192, 8192 + 64 + 3, 300_007, (1 << 21) + 8192 + 77]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ea.init(0)


@pytest.mark.parametrize("f", [static_vbp_f(12, 1), static_vbp_f(1, 1), static_vbp_f(33, 1), static_vbp_f(12, 8),
                               static_vbp_f(64, 8), static_vbp_f(9, 2), dynamic_vbp_f(512, 2048, 8),
                               dynamic_vbp_f(1024, 64, 8), default_for_dynamic_vbp_f(8),
                               default_delta_dynamic_vbp_f(8), rle_f(), uncompr_f()], ids=repr)
@pytest.mark.parametrize("lanes", [1, 8])
def test_select_positions(f, lanes):
    bits = min(f.bw, 40) if f.kind == 1 else 40
    for n in SIZES:
        x = datagen.uniform_bits(0x4D6F7270 + n, n, bits)
        col = ea.morph(f, ea.upload_values(x)) if f.kind else ea.upload_values(x)
        mid = int(x[n // 2]) if n else 3
        for cmp, val in [(MS_CMP_LT, 1 << (bits - 1)), (MS_CMP_EQ, mid), (MS_CMP_NE, mid), (MS_CMP_LT, 0),
                         (MS_CMP_GE, 0)]:
            g = ea.select(cmp, val, uncompr_f(), col, lanes)
            want = rm.select_positions(x, cmp, val)
            m = g.meta()
            assert (m.count, m.size_used, m.size_compr) == (len(want), 8 * len(want), 0), (n, cmp)
            assert np.array_equal(g.values(), want), (n, cmp)


@pytest.mark.parametrize("n", [(1 << 23) + 12345])
def test_select_positions_long(n):
    x = datagen.uniform_bits(5, n, 12)
    for f in (static_vbp_f(12, 1), dynamic_vbp_f(512, 2048, 8), uncompr_f()):
        col = ea.morph(f, ea.upload_values(x)) if f.kind else ea.upload_values(x)
        for cmp, val in [(MS_CMP_LT, 1 << 11), (MS_CMP_EQ, 77)]:
            assert np.array_equal(ea.select(cmp, val, uncompr_f(), col, 8).values(), rm.select_positions(x, cmp, val))


@pytest.mark.parametrize("f", [static_vbp_f(12, 1), dynamic_vbp_f(512, 2048, 8), uncompr_f()], ids=repr)
def test_select_positions_many_tiles(f):
    # 4097 tiles of 32768 rows, several per resident workgroup: its row words
    # and ticket are reused from turn to turn
    n = (1 << 27) + 77
    x = (np.arange(n, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)) >> np.uint64(52)
    col = ea.upload_values(x)
    if f.kind:
        col = ea.morph(f, col)
    for cmp, val in [(MS_CMP_LT, 1 << 11), (MS_CMP_EQ, 77)]:
        assert np.array_equal(ea.select(cmp, val, uncompr_f(), col, 8).values(), rm.select_positions(x, cmp, val))
