"""delta_f of blocks that are no multiple of 512 values, the unit in which
differences are summed: compressed parts that end inside a unit and inside a
tile of 2048, every step, against the oracle and the values themselves."""
import numpy as np
import pytest

import engine_amd as ea
from engine_amd import datagen
from engine_amd.formats import MS_CMP_GE, MS_CMP_LT, delta_f, dynamic_vbp_f, static_vbp_f, uncompr_f
from tests import refmodel as rm

pytestmark = pytest.mark.gpu

FORMATS = [delta_f(64, 1, uncompr_f()), delta_f(192, 1, static_vbp_f(12, 1)), delta_f(128, 2, dynamic_vbp_f(128, 16, 2)),
           delta_f(256, 4, static_vbp_f(12, 4)), delta_f(40, 8, uncompr_f()), delta_f(512, 8, static_vbp_f(12, 8))]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ea.init(0)


@pytest.mark.parametrize("f", FORMATS, ids=repr)
@pytest.mark.parametrize("n", [63, 64, 511, 512, 576, 1344, 2048, 2112, 8191, 300_007])
def test_delta_blocks(oracle, f, n):
    x = datagen.sorted_geometric(n, n)
    g, o = ea.morph(f, ea.upload_values(x)), oracle.morph(f, x)
    img, meta = g.image()
    assert meta == o.meta() and img.tobytes() == o.image().tobytes()
    up = ea.upload_image(f, img, *meta)
    mid = int(x[n // 2])
    for c in (g, up):
        assert np.array_equal(c.values(), x)
        batch, res = ea.Batch(), ea.DeviceU64(2)
        for cmp in (MS_CMP_LT, MS_CMP_GE):
            want = rm.masked_sum(x, cmp, mid)
            assert int(ea.select_sum(cmp, mid, c).get()[0]) == want
            assert int(ea.select_sum_noalloc(cmp, mid, c).get()[0]) == want
            batch.enqueue(c, cmp, mid)
            assert np.array_equal(ea.select(cmp, mid, uncompr_f(), c).values(), rm.select_positions(x, cmp, mid))
        batch.run(res)
        assert res.get().tolist() == [rm.masked_sum(x, cmp, mid) for cmp in (MS_CMP_LT, MS_CMP_GE)]
