"""Memory of the null stream is kept for its next calls: blocks that go from
one call's output to another's scratch, columns read on a created stream
before they are freed, frees from several threads, and frees while a plan
captures leave every result as it was.  What is kept goes back when an
allocation fails, with the last column and on request, and is not what a
non-blocking stream or a plan reads."""
import ctypes
import gc
import threading

import numpy as np
import pytest

import engine_amd as ea
from engine_amd import datagen, hip
from engine_amd.formats import (MS_CMP_GE, MS_CMP_LT, MS_ERR_INVALID, MS_ERR_NOMEM, MS_OP_ADD, blockwise_individual_f,
                                default_delta_dynamic_vbp_f, dynamic_vbp_f, rle_f, uncompr_f)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    ea.init(0)


def below(x, v):
    return int(x[x < v].sum(dtype=np.uint64))


def test_columns_read_on_a_created_stream():
    st, res = hip.Stream(), ea.DeviceU64(40)
    want = []
    for k in range(40):
        x = datagen.uniform_bits(100 + k, 30_000 + 512 * (k % 3), 20)
        col = ea.morph(dynamic_vbp_f(512, 2048, 8), ea.upload_values(x))
        ea.select_sum(MS_CMP_LT, 1 << 19, col, res.at(k), st)
        want.append(below(x, 1 << 19))
        del col         # its block serves the next column while the stream still reads it
    assert res.get().tolist() == want


def test_threads_share_the_null_stream():
    bad = []

    def work(seed):
        ea.init(0)
        for k in range(12):
            n = 5000 + 7001 * (k % 4) + seed
            x = datagen.sorted_geometric(seed + k, n)
            f = (default_delta_dynamic_vbp_f(8), rle_f(), dynamic_vbp_f(512, 64, 8))[k % 3]
            c = ea.morph(f, ea.upload_values(x))
            if not np.array_equal(ea.morph(uncompr_f(), c).values(), x):
                bad.append((seed, k))

    ts = [threading.Thread(target=work, args=(1000 * i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


def test_free_while_a_plan_captures():
    st, plan = hip.Stream(), ea.Plan()
    x = datagen.uniform_bits(3, 50_000, 16)
    col = ea.morph(dynamic_vbp_f(512, 2048, 8), ea.upload_values(x))
    hip.synchronize()
    spare = ea.upload_values(x)
    with plan.record(st):
        ea.agg_sum(col, st)
    with plan.record(st):
        total = ea.agg_sum(col, st)
        del spare       # given back at the end of the capture
    again = ea.upload_values(x ^ np.uint64(1))
    for _ in range(3):
        plan.launch(st)
        st.synchronize()
        assert int(total.values(st)[0]) == int(x.sum(dtype=np.uint64))
        assert np.array_equal(again.values(), x ^ np.uint64(1))
    del total
    plan.free()


def last_error():
    return hip.hip().hipGetLastError()


def used_by_pool():
    """Bytes of the null stream's pool that are allocated (kept ones too)."""
    hip.synchronize()
    pool, used = ctypes.c_void_p(), ctypes.c_uint64()
    assert hip.hip().hipDeviceGetDefaultMemPool(ctypes.byref(pool), 0) == 0
    assert hip.hip().hipMemPoolGetAttribute(pool, 7, ctypes.byref(used)) == 0   # hipMemPoolAttrUsedMemCurrent
    return used.value


@pytest.mark.parametrize("created", [False, True])
def test_failed_allocation(created):
    """An allocation that cannot succeed (2^44 values of one run) gives the
    kept memory back, is an error of its own call and of no later one."""
    st = hip.Stream() if created else None
    pair = np.array([7, 1 << 44], np.uint64).view(np.uint8)
    run = ea.upload_image(rle_f(), pair, 1 << 44, 16, 16)
    x = datagen.uniform_bits(9, 1 << 20, 20)
    left = []
    for _ in range(2):
        ea.upload_values(x)                   # freed at once: 8 MiB kept
        kept = used_by_pool()
        with pytest.raises(ea.MsError) as e:
            ea.morph(uncompr_f(), run, st)
        assert e.value.code == MS_ERR_NOMEM
        assert last_error() == 0
        left.append(used_by_pool())
        assert left[-1] <= kept - x.nbytes
    assert left[0] == left[1]
    assert np.array_equal(ea.morph(dynamic_vbp_f(512, 2048, 8), ea.upload_values(x), st).values(st), x)


def test_failed_plan_arena():
    x = datagen.uniform_bits(9, 1 << 20, 20)
    keep = ea.upload_values(x[:10])
    ea.upload_values(x)
    kept = used_by_pool()
    with pytest.raises(ea.MsError) as e:
        ea.Plan(1 << 46)
    assert e.value.code == MS_ERR_NOMEM
    assert last_error() == 0 and used_by_pool() <= kept - x.nbytes
    assert np.array_equal(keep.values(), x[:10])


def test_release_memory():
    x = datagen.uniform_bits(9, 1 << 20, 20)
    keep = ea.upload_values(x[:10])
    ea.release_memory()
    before = used_by_pool()
    ea.upload_values(x)
    assert used_by_pool() >= before + x.nbytes
    ea.release_memory()
    assert used_by_pool() == before
    assert np.array_equal(keep.values(), x[:10])


def test_release_memory_not_while_a_plan_captures():
    st, plan = hip.Stream(), ea.Plan()
    col = ea.upload_values(datagen.uniform_bits(9, 5000, 20))
    with plan.record(st):
        ea.agg_sum(col, st)
    with plan.record(st):
        with pytest.raises(ea.MsError) as e:
            ea.release_memory()
        total = ea.agg_sum(col, st)
    assert e.value.code == MS_ERR_INVALID
    plan.launch(st)
    assert int(total.values(st)[0]) == int(col.values().sum(dtype=np.uint64))
    del total
    plan.free()


@pytest.mark.parametrize("make", [lambda n: ea.DeviceU64(n), lambda n: hip.DeviceArray(n, np.uint64)])
def test_failed_device_array(make):
    x = datagen.uniform_bits(9, 1 << 20, 20)
    keep = ea.upload_values(x[:10])
    ea.upload_values(x)
    kept = used_by_pool()
    with pytest.raises(RuntimeError):
        make(1 << 43)
    assert last_error() == 0 and used_by_pool() <= kept - x.nbytes
    assert np.array_equal(keep.values(), x[:10])


def test_nothing_is_kept_without_columns():
    """The last column's free gives everything back, also if that column is a
    plan's."""
    gc.collect()
    x = datagen.uniform_bits(9, 1 << 20, 20)
    keep = ea.upload_values(x[:10])
    ea.release_memory()
    before = used_by_pool()
    st, plan = hip.Stream(), ea.Plan()
    with plan.record(st):
        ea.agg_sum(keep, st)
    with plan.record(st):
        total = ea.agg_sum(keep, st)
    ea.upload_values(x)
    del keep
    assert used_by_pool() >= before + x.nbytes - 8192
    del total                                 # the last column
    assert used_by_pool() < before
    plan.free()


class NonBlocking:
    """A created stream that the null stream does not wait for."""

    def __init__(self):
        self._as_parameter_ = ctypes.c_void_p()
        assert hip.hip().hipStreamCreateWithFlags(ctypes.byref(self._as_parameter_), 1) == 0

    def synchronize(self):
        assert hip.hip().hipStreamSynchronize(self._as_parameter_) == 0

    def destroy(self):
        assert hip.hip().hipStreamDestroy(self._as_parameter_) == 0


D = dynamic_vbp_f(512, 2048, 8)


def batch_run(col, pos, st, res):
    b = ea.Batch()
    b.enqueue(col, MS_CMP_LT, 9)
    b.run(res, st)
    return b


READS = {
    "select_sum": lambda col, pos, st, res: ea.select_sum(MS_CMP_LT, 9, col, res, st),
    "select_sum_noalloc": lambda col, pos, st, res: ea.select_sum_noalloc(MS_CMP_LT, 9, col, res, st),
    "morph": lambda col, pos, st, res: ea.morph(D, col, st),
    "morph_blockwise": lambda col, pos, st, res: ea.morph_blockwise(blockwise_individual_f(1024), col,
                                                                    np.full(1024, 65, np.uint8), st),
    "select": lambda col, pos, st, res: ea.select(MS_CMP_LT, 9, uncompr_f(), col, 8, st),
    "between": lambda col, pos, st, res: ea.between(MS_CMP_GE, 2, MS_CMP_LT, 9, uncompr_f(), col, 8, st),
    "project_data": lambda col, pos, st, res: ea.project(uncompr_f(), col, pos, 8, st),
    "project_pos": lambda col, pos, st, res: ea.project(uncompr_f(), col, col, 8, st),
    "agg_sum": lambda col, pos, st, res: ea.agg_sum(col, st),
    "intersect_l": lambda col, pos, st, res: ea.intersect_sorted(uncompr_f(), col, pos, st),
    "intersect_r": lambda col, pos, st, res: ea.intersect_sorted(uncompr_f(), pos, col, st),
    "merge_l": lambda col, pos, st, res: ea.merge_sorted(uncompr_f(), col, pos, st),
    "merge_r": lambda col, pos, st, res: ea.merge_sorted(uncompr_f(), pos, col, st),
    "calc": lambda col, pos, st, res: ea.calc_binary(MS_OP_ADD, uncompr_f(), col, col, st),
    "group": lambda col, pos, st, res: ea.group(uncompr_f(), uncompr_f(), col, None, st),
    "group_of": lambda col, pos, st, res: ea.group(uncompr_f(), uncompr_f(), col, col, st),
    "join": lambda col, pos, st, res: ea.join(uncompr_f(), uncompr_f(), pos, col, st),
    "semi_join": lambda col, pos, st, res: ea.semi_join(uncompr_f(), pos, col, st),
    "batch": batch_run,
}


@pytest.mark.parametrize("op", READS)
def test_columns_read_on_a_non_blocking_stream(op):
    """They go to the pool: the null stream's next call does not wait for
    such a stream.  Read on a blocking one they are kept."""
    for st, kept in ((NonBlocking(), False), (hip.Stream(), True)):
        res = ea.DeviceU64()
        pos = ea.upload_values(np.arange(40, dtype=np.uint64))
        ea.release_memory()
        before = used_by_pool()
        col = ea.upload_values(np.arange(1 << 20, dtype=np.uint64))
        hip.synchronize()
        out = READS[op](col, pos, st, res)
        st.synchronize()
        del out
        del col
        assert (used_by_pool() >= before + (8 << 20)) == kept
        if not kept:
            st.destroy()


def test_columns_read_by_a_plan():
    """A plan may be launched on any stream."""
    st, plan = hip.Stream(), ea.Plan()
    keep = ea.upload_values(np.arange(40, dtype=np.uint64))
    ea.release_memory()
    before = used_by_pool()
    col = ea.upload_values(np.arange(1 << 20, dtype=np.uint64))
    hip.synchronize()
    with plan.record(st):
        ea.agg_sum(col, st)
    with plan.record(st):
        total = ea.agg_sum(col, st)
    plan.launch(st)
    assert int(total.values(st)[0]) == (1 << 19) * ((1 << 20) - 1)
    del total
    plan.free()
    del col
    assert used_by_pool() < before + (8 << 20)
    assert len(keep.values()) == 40


def test_freed_while_a_plan_captures_after_a_non_blocking_read():
    nb, res = NonBlocking(), ea.DeviceU64()
    st, plan = hip.Stream(), ea.Plan()
    keep = ea.upload_values(np.arange(40, dtype=np.uint64))
    with plan.record(st):
        ea.agg_sum(keep, st)
    ea.release_memory()
    before = used_by_pool()
    col = ea.upload_values(np.arange(1 << 20, dtype=np.uint64))
    hip.synchronize()
    ea.select_sum(MS_CMP_LT, 9, col, res, nb)
    nb.synchronize()
    with plan.record(st):
        total = ea.agg_sum(keep, st)
        del col
    assert used_by_pool() < before + (8 << 20)
    plan.launch(st)
    assert int(total.values(st)[0]) == 780 and int(res.get()[0]) == 36
    del total
    plan.free()
    nb.destroy()
