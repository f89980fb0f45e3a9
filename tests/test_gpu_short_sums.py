"""Fused select + sum and agg_sum of short columns (one workgroup, no partial
sums) and of those just beyond: every layout, with and without a raw rest,
results and metas as for long columns."""
import numpy as np
import pytest

import engine_amd as ea
from engine_amd import datagen
from engine_amd.formats import (MS_CMP_EQ, MS_CMP_GE, MS_CMP_LT, MS_CMP_NE, default_delta_dynamic_vbp_f,
                                default_for_dynamic_vbp_f, delta_f, dynamic_vbp_f, for_f, rle_f, static_vbp_f,
                                uncompr_f)
from tests import refmodel as rm

pytestmark = pytest.mark.gpu

FORMATS = [uncompr_f(), static_vbp_f(20, 1), static_vbp_f(20, 8), static_vbp_f(20, 3), dynamic_vbp_f(512, 2048, 8),
           dynamic_vbp_f(64, 8, 1), for_f(512, 8, uncompr_f()), default_delta_dynamic_vbp_f(8),
           delta_f(1024, 8, static_vbp_f(40, 8)), default_for_dynamic_vbp_f(8), rle_f()]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ea.init(0)


@pytest.mark.parametrize("f", FORMATS, ids=repr)
@pytest.mark.parametrize("n", [0, 1, 511, 513, 2048, 4096, 4097, 6143, 8191, 8192, 8193, 12_345])
def test_short_sums(oracle, f, n):
    x = datagen.uniform_bits(0x4D6F7270 + n, n, 20)
    if f.kind == 3:
        x = np.sort(x)
    col = ea.morph(f, ea.upload_values(x)) if f.kind else ea.upload_values(x)
    mid = int(x[n // 2]) if n else 7
    for cmp, val in [(MS_CMP_LT, mid), (MS_CMP_EQ, mid), (MS_CMP_NE, mid), (MS_CMP_GE, 0), (MS_CMP_LT, 0)]:
        want = rm.masked_sum(x, cmp, val)
        assert int(ea.select_sum(cmp, val, col).get()[0]) == want
        assert int(ea.select_sum_noalloc(cmp, val, col).get()[0]) == want
    g, o = ea.agg_sum(col), oracle.agg_sum(oracle.morph(f, x))
    img, meta = g.image()
    assert meta == o.meta() and img.tobytes() == o.image().tobytes()
