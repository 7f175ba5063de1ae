"""Host arrays to the device and back through pinned memory: lengths around the staging pieces (16 KB per workgroup, 256 KB for
a call's first piece, 1 MB slots, 8 of them before one is used again), conversions bit for bit numpy's, streams and threads."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 5, 4095, 4096, 4097, 65535, 65537, 262143, 300001, 5 * 262144 + 7])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "i32"])
def test_round_trip_of_every_length(lm, hip, oracle, n, dtype):
    x = oracle.gen_normal((n,), 41000 + n) * np.float32(1000) if dtype != "i32" else np.arange(n, dtype=np.int32) * 7919 - 5
    got = lm.to_device(x, hip, dtype).to_host()
    np.testing.assert_array_equal(got, x if dtype == "i32" else lm.decode(lm.encode(x, dtype), dtype))
    assert got.flags.writeable and got.flags.c_contiguous


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_conversions_at_the_ends_of_the_range(lm, hip, dtype):
    x = np.array([0.0, -0.0, np.inf, -np.inf, 65504, 65519, 65520, 1e-8, 6e-8, 3e-5, -6.1e-5, 3.4e38, 1e-40, 1.00390625, 1.01171875, 2049, 2051], np.float32)
    raw = lm.HipArray(x.shape, dtype, hip).copy_from_host(x).to_host_raw()
    np.testing.assert_array_equal(raw.view(np.uint16), lm.encode(x, dtype).view(np.uint16))
    assert np.isnan(lm.HipArray((1,), dtype, hip).copy_from_host(np.array([np.nan], np.float32)).to_host()[0])


def test_many_uploads_reuse_the_slots_in_order(lm, hip):
    # 40 arrays of 0.9 MB on the null stream and on another one: every slot is used several times
    b, stream = lm.binding, lm.binding.stream_create()
    host = [np.full(225000, i, np.float32) for i in range(40)]
    dev = [lm.HipArray((225000,), "f16" if i % 3 == 0 else "f32", hip) for i in range(40)]
    for i, (d, h) in enumerate(zip(dev, host)):
        b.upload([d._upload_item(h)[0]], stream if i % 4 == 1 else None)
        h[:] = -1  # the host memory may be reused at once
    b.sync(stream)
    b.sync()
    b.stream_destroy(stream)
    for i, d in enumerate(dev):
        got = d.to_host()
        assert got[0] == i and got[-1] == i and (got == i).all()


def test_threads_that_execute_at_the_same_time(lm, hip, oracle):
    g = lm.Graph()
    q, k, v = (lm.tensor(g, (1, 4, 200, 64)) for _ in range(3))
    out = lm.flash_attention(q, k, v, causal=True)
    feeds = [{t.id: oracle.gen_normal((1, 4, 200, 64), 42000 + 10 * j + i) for i, t in enumerate((q, k, v))} for j in range(4)]
    want = [lm.execute(g, out.id, f, hip) for f in feeds]
    wrong = []

    def work(j):
        for _ in range(10):
            if not np.array_equal(lm.execute(g, out.id, feeds[j], hip), want[j]):
                wrong.append(j)

    threads = [threading.Thread(target=work, args=(j,)) for j in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not wrong


def test_results_stay_theirs_and_the_pools_are_given_back(lm, hip):
    a = lm.to_device(np.arange(5000, dtype=np.float32), hip)
    kept = [a.to_host() for _ in range(5)]  # five live arrays: five blocks
    kept[0][:] = 0
    np.testing.assert_array_equal(kept[1], np.arange(5000, dtype=np.float32))
    assert len({x.ctypes.data for x in kept}) == 5
    del kept
    pool = lm.host._pinned
    assert pool.kept > 0
    lm.release_pools()
    assert pool.kept == 0 and all(p.kept == 0 for p in lm.host._device_pools.values())
    most, pool.most = pool.most, pool.used  # nothing more to be had: an ordinary array
    try:
        np.testing.assert_array_equal(a.to_host(), np.arange(5000, dtype=np.float32))
    finally:
        pool.most = most


@pytest.mark.parametrize("n,src_at,dst_at", [(1, 0, 0), (4097, 1, 0), (4098, 0, 1), (300001, 3, 2), (300001, 0, 0)])
def test_fp32_downloads_of_any_alignment(lm, hip, oracle, n, src_at, dst_at):
    """By a kernel where the ends are aligned and pinned, otherwise by the runtime: into pinned memory at any float, and into pageable."""
    b = lm.binding
    x = oracle.gen_normal((n + 8,), 43000 + n)
    x[src_at] = np.float32(1e-45)  # the smallest subnormal stays what it is
    dev = lm.to_device(x, hip)
    ptr = b.host_alloc(4 * (n + 8))
    pinned = np.frombuffer((ctypes.c_char * (4 * (n + 8))).from_address(ptr), np.float32)
    pageable = np.empty(n + 8, np.float32)
    for to, at in ((pinned, ptr), (pageable, pageable.ctypes.data)):
        to[:] = -7
        b.download(at + 4 * dst_at, dev.ptr + 4 * src_at, n, b.LMH_F32)
        b.sync()
        np.testing.assert_array_equal(to[dst_at:dst_at + n], x[src_at:src_at + n])
        assert (to[:dst_at] == -7).all() and (to[dst_at + n:] == -7).all()
    del pinned, to
    b.host_free(ptr)
