"""What compile() and execute() make of the nodes around attention, on host memory (host_device.py)."""
import gc

import numpy as np
import pytest

from host_device import HostDevice


@pytest.fixture
def mem(lm, monkeypatch):
    device = HostDevice(lm)
    device.hip = device.install(monkeypatch)
    yield device
    gc.collect()


def normal(shape, seed):
    return np.random.default_rng(seed).standard_normal(shape).astype(np.float32)


def close(got, want):
    np.testing.assert_allclose(got, want, rtol=2e-6, atol=2e-6)


# ---- declared shapes -------------------------------------------------------------------------
def test_a_fed_array_of_another_size_is_refused(lm, mem):
    g = lm.Graph()
    x = lm.tensor(g, (1, 16, 64))
    layer = lm.Linear(64, 32, g, bias=False)
    out = layer(x)
    y = lm.tensor(g, (4, 8))
    moved = lm.permute(y, (1, 0))
    w = normal((32, 64), 1)
    with pytest.raises(ValueError):
        lm.execute(g, out.id, {x.id: normal((1, 32, 64), 2), layer.weight.id: w, y.id: normal((4, 8), 3)}, mem.hip)
    with pytest.raises(ValueError):
        lm.execute(g, moved.id, {x.id: normal((1, 16, 64), 2), layer.weight.id: w, y.id: normal((2, 3), 3)}, mem.hip)
    # the same elements under another shape are taken as they lie
    a = normal((8, 4), 4)
    got = lm.execute(g, moved.id, {x.id: normal((16, 64), 2), layer.weight.id: w, y.id: a}, mem.hip)
    np.testing.assert_array_equal(got, a.reshape(4, 8).T)


def test_a_node_declared_in_another_shape_than_its_op_gives_stays_out_of_launches(lm, mem):
    # add_op takes any shape: the op's own result decides, as it does for a node that runs alone
    def graph(shape):
        g = lm.Graph()
        x, w = lm.tensor(g, (2, 6, 8)), lm.tensor(g, (5, 8))
        product = lm.matmul(x, lm.permute(w, (1, 0)))
        g.shapes[product.id] = shape
        return g, x, w, product

    a, b = normal((2, 6, 8), 1), normal((5, 8), 2)
    for shape in ((2, 3, 5), (2, 6, 4), (1, 1, 1)):
        g, x, w, product = graph(shape)
        close(lm.execute(g, product.id, {x.id: a, w.id: b}, mem.hip), a @ b.T)
        with pytest.raises(ValueError):
            lm.compile(g, mem.hip)({x.id: a, w.id: b})
    for shape in ((2, 2), (8, 4, 2)):
        g = lm.Graph()
        x = lm.tensor(g, (4, 8))
        y = lm.add_op(g, lm.PermuteOp((1, 0)), [(x.id, 0, (4, 8))], shape)
        c = normal((4, 8), 3)
        np.testing.assert_array_equal(lm.execute(g, y.id, {x.id: c}, mem.hip), c.T)
        with pytest.raises(ValueError):
            lm.compile(g, mem.hip)({x.id: c})


def test_weights_read_under_another_shape(lm, mem):
    # W^T's elements as a (16, 4) matrix: not a product with W as it lies
    g = lm.Graph()
    x, w = lm.tensor(g, (1, 3, 16)), lm.tensor(g, (8, 8))
    wt = lm.permute(w, (1, 0))
    wt.shape = (16, 4)
    out = lm.matmul(x, wt)
    a, b = normal((1, 3, 16), 1), normal((8, 8), 2)
    close(lm.execute(g, out.id, {x.id: a, w.id: b}, mem.hip), a @ np.ascontiguousarray(b.T).reshape(16, 4))
    cg = lm.compile(g, mem.hip)
    close(cg({x.id: a, w.id: b})[out.id].to_host(), a @ np.ascontiguousarray(b.T).reshape(16, 4))


def test_a_chain_of_more_dimensions_than_a_launch_takes(lm, mem):
    g = lm.Graph()
    x = lm.tensor(g, (512,))
    split = lm.reshape(x, (2,) * 9)
    out = lm.permute(split, (1, 0, 3, 2, 5, 4, 7, 6, 8)[::-1])
    a = normal((512,), 1)
    want = g.nodes[out.id].op.compute(g.nodes[split.id].op.compute(a))
    np.testing.assert_array_equal(lm.execute(g, out.id, {x.id: a}, mem.hip), want)
    np.testing.assert_array_equal(lm.compile(g, mem.hip)({x.id: a})[out.id].to_host(), want)


# ---- nodes that write into their inputs ------------------------------------------------------
def cache_graph(lm, before, after):
    """before(k cache) -> append a row -> after(what before gave); (graph, feeds, tensors by name)."""
    g = lm.Graph()
    kc, vc = lm.tensor(g, (2, 1, 4, 6)), lm.tensor(g, (2, 1, 4, 6))
    kn, vn, pos = lm.tensor(g, (2, 1, 1, 6)), lm.tensor(g, (2, 1, 1, 6)), lm.tensor(g, (2,), "i32")
    first = before(kc)
    k2, v2 = lm.kv_cache_append(kc, vc, kn, vn, pos)
    last = after(first, k2)
    feeds = {kc.id: normal((2, 1, 4, 6), 1), vc.id: normal((2, 1, 4, 6), 2), kn.id: normal((2, 1, 1, 6), 3), vn.id: normal((2, 1, 1, 6), 4),
             pos.id: np.array([3, 1], np.int32)}
    return g, feeds, kc.id, first.id, last.id


def test_a_chain_reads_its_operand_before_it_is_written(lm, mem):
    g, feeds, kc, first, last = cache_graph(lm, lambda k: lm.permute(k, (0, 1, 3, 2)), lambda x, k2: lm.permute(x, (2, 3, 0, 1)))
    want = feeds[kc].transpose(0, 1, 3, 2).transpose(2, 3, 0, 1)
    np.testing.assert_array_equal(lm.execute(g, last, feeds, mem.hip), want)
    cg = lm.compile(g, mem.hip)
    for _ in range(2):
        np.testing.assert_array_equal(cg(feeds)[last].to_host(), want)


def test_a_node_asked_for_has_the_value_from_before_a_later_write(lm, mem):
    g, feeds, kc, first, last = cache_graph(lm, lambda k: lm.permute(lm.permute(k, (0, 1, 3, 2)), (2, 3, 0, 1)), lambda x, k2: lm.permute(k2, (0, 2, 1, 3)))
    cg = lm.compile(g, mem.hip)
    for _ in range(2):
        res = cg(feeds)
        np.testing.assert_array_equal(res[first].to_host(), feeds[kc].transpose(0, 1, 3, 2).transpose(2, 3, 0, 1))
        np.testing.assert_array_equal(res[first - 1].to_host(), feeds[kc].transpose(0, 1, 3, 2))


def test_products_with_weights_that_are_written_later(lm, mem):
    g = lm.Graph()
    kc, vc = lm.tensor(g, (1, 1, 4, 6)), lm.tensor(g, (1, 1, 4, 6))
    kn, vn, pos, x = lm.tensor(g, (1, 1, 1, 6)), lm.tensor(g, (1, 1, 1, 6)), lm.tensor(g, (1,), "i32"), lm.tensor(g, (1, 3, 6))
    w = lm.GraphTensor(kc.id, (4, 6), g)
    wt = lm.permute(w, (1, 0))
    lm.kv_cache_append(kc, vc, kn, vn, pos)
    out = lm.matmul(x, wt)
    feeds = {kc.id: normal((1, 1, 4, 6), 1), vc.id: normal((1, 1, 4, 6), 2), kn.id: normal((1, 1, 1, 6), 3), vn.id: normal((1, 1, 1, 6), 4),
             pos.id: np.array([2], np.int32), x.id: normal((1, 3, 6), 5)}
    want = feeds[x.id] @ feeds[kc.id][0, 0].T
    close(lm.execute(g, out.id, feeds, mem.hip), want)
    cg = lm.compile(g, mem.hip)
    for _ in range(2):
        close(cg(feeds)[out.id].to_host(), want)
        np.testing.assert_array_equal(cg.results[wt.id].to_host(), feeds[kc.id][0, 0].T)


# ---- nodes computed when they are asked for --------------------------------------------------
def test_a_node_asked_for_comes_after_its_operand(lm, mem):
    g = lm.Graph()
    x, c, w, bias = lm.tensor(g, (2, 3, 4)), lm.tensor(g, (4,)), lm.tensor(g, (4, 4)), lm.tensor(g, (4,))
    lm.add(x, c)
    product = lm.matmul(x, lm.permute(w, (1, 0)))
    plus = lm.add(x, c)
    inner = lm.permute(plus, (0, 2, 1))
    outer = lm.permute(inner, (2, 1, 0))
    for _ in range(3):
        outer = lm.add(outer, lm.tensor(g, (1,)))
    # the product's launch stands for its last node, the one with the highest number
    out = lm.add(product, lm.expand(lm.expand(bias, 0, 3), 0, 2))
    values = {i: normal(g.shapes[i], 50 + i) for i, n in enumerate(g.nodes) if isinstance(n.op, lm.host.InputTensor)}
    cg = lm.compile(g, mem.hip)
    cg(values)
    handed = cg.results[inner.id]
    for seed in (1, 2):
        values[x.id] = normal((2, 3, 4), seed)
        res = cg(values)
        np.testing.assert_array_equal(handed.to_host(), (values[x.id] + values[c.id]).transpose(0, 2, 1))
        assert res[inner.id] is handed
        close(res[out.id].to_host(), values[x.id] @ values[w.id].T + values[bias.id])


@pytest.mark.parametrize("seed", range(40))
def test_every_node_of_random_graphs(lm, mem, seed):
    """Views, sums, products and cache appends in random order: the value of every node, asked for in random order, after each
    of several calls, is what the nodes one by one give."""
    rng = np.random.default_rng(seed)
    g = lm.Graph()
    B, S, W = 2, 4, 6
    shape = (B, S, W)
    pool = [lm.tensor(g, shape) for _ in range(2)]
    caches = [lm.tensor(g, (B, 1, S, W)) for _ in range(2)]
    pos, weights, bias = lm.tensor(g, (B,), "i32"), [lm.tensor(g, (W, W)) for _ in range(2)], lm.tensor(g, (W,))
    for _ in range(12):
        a = pool[rng.integers(len(pool))]
        kind = rng.integers(7)
        if kind <= 1:
            a = lm.permute(a, tuple(int(d) for d in rng.permutation(3)))
        elif kind == 2:
            a = lm.reshape(a, [(B, S, W), (S, B, W), (W, S, B), (B, W, S)][rng.integers(4)])
        elif kind == 3 and a.shape == shape:
            a = lm.add(a, pool[0])
        elif kind == 4 and a.shape == shape:
            a = lm.matmul(a, lm.permute(weights[rng.integers(2)], (1, 0)))
            if rng.integers(2):
                a = lm.add(a, lm.expand(lm.expand(bias, 0, S), 0, B))
            if rng.integers(2):
                a = lm.permute(lm.reshape(a, (B, S, 3, 2)), (0, 2, 1, 3))
                a = lm.reshape(lm.permute(a, (0, 2, 1, 3)) if rng.integers(2) else a, shape)
        elif kind == 5:
            new = [lm.GraphTensor(t.id, (B, 1, 2, W), g, t.index) for t in (lm.tensor(g, (B, 2, W)), lm.tensor(g, (B, 2, W)))]
            lm.kv_cache_append(caches[0], caches[1], new[0], new[1], pos)
            continue
        else:
            cache = caches[rng.integers(2)]
            a = lm.GraphTensor(cache.id, shape, g)
        pool.append(a)
    inputs = [i for i, n in enumerate(g.nodes) if isinstance(n.op, lm.host.InputTensor)]

    def feeds():
        return {i: rng.integers(0, S - 1, B).astype(np.int32) if i == pos.id else rng.standard_normal(g.shapes[i]).astype(np.float32) for i in inputs}

    def one_by_one(values):
        got = {i: v.copy() for i, v in values.items()}
        pick = lambda r: np.ascontiguousarray(got[r[0]]).reshape(r[2])
        for i, n in enumerate(g.nodes):
            if i in got:
                continue
            if isinstance(n.op, lm.KVAppendOp):
                for b, p in enumerate(values[pos.id]):
                    for cache, new in zip(n.inputs[:2], n.inputs[2:4]):
                        got[cache[0]][b, :, p:p + 2] = pick(new)[b]
            else:
                got[i] = np.array(n.op.compute(*[pick(r) for r in n.inputs]), np.float32)
        return got

    def same(got, want):  # up to 12 nodes in fp32, each within a few roundings of its largest term
        np.testing.assert_allclose(got, want, rtol=0, atol=12 * 6 * 2.0 ** -24 * max(1.0, float(np.abs(want).max())) * W)

    cg = lm.compile(g, mem.hip)
    asked = []
    nodes = [i for i, n in enumerate(g.nodes) if not isinstance(n.op, lm.KVAppendOp)]
    for _ in range(3):
        values = feeds()
        want = one_by_one(values)
        res = cg(values)
        for i in asked:
            same(res[i].to_host(), want[i])
        asked = [int(i) for i in rng.permutation(nodes)[:6]]
        for i in asked:
            same(res[i].to_host(), want[i])
    for i in nodes[-3:]:
        if i not in inputs:
            same(lm.execute(g, i, values, mem.hip), want[i])


def test_whole_numbers_are_moved_and_multiplied(lm, mem):
    g = lm.Graph()
    x, a, b = lm.tensor(g, (2, 6), "i32"), lm.tensor(g, (3, 4)), lm.tensor(g, (5, 4))
    moved = lm.permute(lm.reshape(lm.expand(x, 0, 2), (4, 6)), (1, 0))
    product = lm.matmul(a, lm.permute(b, (1, 0)), dtype="i32")
    one = lm.reshape(x, (3, 4))
    values = {x.id: np.arange(12, dtype=np.int32).reshape(2, 6) * 1000003 % 16777213, a.id: np.arange(12, dtype=np.float32).reshape(3, 4),
              b.id: np.arange(20, dtype=np.float32).reshape(5, 4) - 7}
    want = {moved.id: np.reshape(np.repeat(values[x.id][None], 2, 0), (4, 6), order="F").T, product.id: values[a.id] @ values[b.id].T,
            one.id: np.reshape(values[x.id], (3, 4), order="F")}
    res = lm.compile(g, mem.hip)(values)
    for i, w in want.items():
        got = lm.execute(g, i, values, mem.hip)
        assert got.dtype == np.int32
        np.testing.assert_array_equal(got, w)
        np.testing.assert_array_equal(res[i].to_host(), w)
    x_dev = lm.to_device(values[x.id], mem.hip)
    op = lm.PermuteOp((1, 0))
    op.out_dtype = "i32"
    np.testing.assert_array_equal(lm.execute_op(op, x_dev).to_host(), values[x.id].T)


# ---- inputs ----------------------------------------------------------------------------------
def test_nothing_is_kept_of_the_arrays_a_call_is_fed(lm, mem):
    g = lm.Graph()
    a, b = lm.tensor(g, (8,)), lm.tensor(g, (8,))
    out = lm.add(a, b)
    cg = lm.compile(g, mem.hip)
    state = set()
    for seed in range(200):
        va, vb = normal((8,), seed), normal((8,), seed + 1000)
        fed = {a.id: lm.to_device(va, mem.hip), b.id: lm.to_device(vb, mem.hip)}
        mem.calls.clear()
        np.testing.assert_array_equal(cg(fed)[out.id].to_host(), va + vb)
        assert mem.calls == ["copy_many 2", "map"]
        state.add(repr({k: sorted(map(str, v)) if isinstance(v, dict) else str(v) for k, v in vars(cg).items()}))
    assert len(state) == 1  # the graph after 200 calls with arrays of their own is the graph after one
    assert all(addr not in repr([list(cg._copies.dst), cg._copies.nodes]) for addr in (str(x.ptr) for x in fed.values()))
    # other nodes than before, another order, host arrays among them, a wrong length
    np.testing.assert_array_equal(cg({b.id: lm.to_device(va, mem.hip)})[out.id].to_host(), va + va)
    np.testing.assert_array_equal(cg({b.id: lm.to_device(vb, mem.hip), a.id: va})[out.id].to_host(), va + vb)
    with pytest.raises(ValueError, match="node %d" % b.id):
        cg({a.id: lm.to_device(va, mem.hip), b.id: lm.to_device(normal((9,), 1), mem.hip)})
    with pytest.raises(KeyError):
        cg({17: lm.to_device(va, mem.hip)})
    np.testing.assert_array_equal(cg({})[out.id].to_host(), va + vb)


# ---- the kept lowering -----------------------------------------------------------------------
def test_a_changed_graph_is_lowered_again(lm, mem):
    g = lm.Graph()
    x, y = lm.tensor(g, (4, 8)), lm.tensor(g, (4, 8))
    moved = lm.permute(lm.permute(x, (1, 0)), (1, 0))
    out = lm.permute(moved, (1, 0))
    feeds = {x.id: normal((4, 8), 1), y.id: normal((4, 8), 2)}

    def value():
        return lm.execute(g, out.id, feeds, mem.hip)

    np.testing.assert_array_equal(value(), feeds[x.id].T)
    g.nodes[moved.id - 1].inputs = [(y.id, 0, (4, 8))]  # another operand
    np.testing.assert_array_equal(value(), feeds[y.id].T)
    g.nodes[out.id].op.dims = (0, 1)  # another op
    g.shapes[out.id] = (4, 8)
    np.testing.assert_array_equal(value(), feeds[y.id])
    g.dtypes[out.id] = g.nodes[out.id].op.out_dtype = "f16"  # another type
    np.testing.assert_array_equal(value(), feeds[y.id].astype(np.float16).astype(np.float32))
    kept = g.lowered([out.id], feeds)
    assert g.lowered([out.id], feeds) is kept


def test_threads_lower_a_new_graph_at_the_same_time(lm, mem):
    import random
    import threading
    import time

    class SlowGraph(lm.Graph):  # every access to what is kept takes its time
        def __init__(self):
            self.kept = None
            super().__init__()

        @property
        def _lowered(self):
            time.sleep(random.uniform(0, 2e-4))
            return self.kept

        @_lowered.setter
        def _lowered(self, value):
            time.sleep(random.uniform(0, 4e-4))
            self.kept = value

    wrong = []
    for _ in range(60):
        g = SlowGraph()
        nodes = [lm.tensor(g, (2, 3))]
        for _ in range(4):
            nodes.append(lm.permute(nodes[-1], (1, 0)))

        def work(wanted):
            try:
                assert g.lowered([wanted], [0])[0][-1].nodes
            except Exception as e:
                wrong.append(repr(e))

        threads = [threading.Thread(target=work, args=(i,)) for i in range(1, 5)]
        [t.start() for t in threads]
        [t.join() for t in threads]
    assert not wrong, wrong[:3]


def test_arrays_of_another_gpu_take_the_runtimes_copy(lm, mem):
    g = lm.Graph()
    a, b = lm.tensor(g, (8,)), lm.tensor(g, (8,))
    out = lm.add(a, b)
    cg = lm.compile(g, mem.hip)
    va, vb = normal((8,), 1), normal((8,), 2)
    fed = {a.id: lm.to_device(va, mem.hip), b.id: lm.to_device(vb, lm.HIPDevice(1))}
    mem.calls.clear()
    np.testing.assert_array_equal(cg(fed)[out.id].to_host(), va + vb)
    assert mem.calls == ["memcpy_d2d", "memcpy_d2d", "map"]
    mem.calls.clear()
    np.testing.assert_array_equal(lm.execute_op(lm.AddOp(), *fed.values()).to_host(), va + vb)  # through the host
    assert mem.calls == []
    h = lm.Graph()
    x = lm.tensor(h, (2, 4))
    moved = lm.permute(x, (1, 0))
    np.testing.assert_array_equal(lm.execute(h, moved.id, {x.id: fed[b.id].view((2, 4))}, mem.hip), vb.reshape(2, 4).T)
    assert mem.calls == ["memcpy_d2d", "map"]


def test_without_a_device_nodes_are_refused_by_name(lm):
    g = lm.Graph()
    x = lm.tensor(g, (2, 4))
    moved = lm.permute(x, (1, 0))
    with pytest.raises(TypeError, match="PermuteOp: no input is on a HIP device"):
        lm.execute(g, moved.id, {x.id: normal((2, 4), 1)}, lm.CPUDevice())


def test_device_arrays_run_where_they_are(lm, mem):
    g = lm.Graph()
    x = lm.tensor(g, (2, 4))
    moved = lm.permute(lm.permute(x, (1, 0)), (1, 0))
    a = normal((2, 4), 1)
    np.testing.assert_array_equal(lm.execute(g, moved.id, {x.id: lm.to_device(a, mem.hip)}, lm.CPUDevice()), a)


def test_views_behind_a_product_that_is_split_into_heads(lm, mem):
    g = lm.Graph()
    x, w = lm.tensor(g, (2, 3, 4)), lm.tensor(g, (8, 4))
    product = lm.matmul(x, lm.permute(w, (1, 0)))
    heads = lm.permute(lm.reshape(product, (2, 3, 2, 4)), (0, 2, 1, 3))
    moved = lm.permute(heads, (3, 0, 1, 2))
    values = {x.id: normal(x.shape, 1), w.id: normal(w.shape, 2)}
    split = np.reshape(values[x.id] @ values[w.id].T, (2, 3, 2, 4), order="F").transpose(0, 2, 1, 3)
    cg = lm.compile(g, mem.hip)
    for _ in range(2):
        res = cg(values)
        close(res[moved.id].to_host(), split.transpose(3, 0, 1, 2))
        close(res[heads.id].to_host(), split)
    close(lm.execute(g, moved.id, values, mem.hip), split.transpose(3, 0, 1, 2))


def test_a_walk_over_all_results_leaves_the_graph_as_it_was(lm, mem):
    g = lm.Graph()
    x, w, b = lm.tensor(g, (2, 3, 4)), lm.tensor(g, (8, 4)), lm.tensor(g, (8,))
    product = lm.matmul(x, lm.permute(w, (1, 0)))
    biased = lm.add(product, lm.expand(lm.expand(b, 0, 3), 0, 2))
    out = lm.permute(lm.reshape(biased, (2, 3, 2, 4)), (0, 2, 1, 3))
    moved = lm.permute(lm.permute(out, (3, 0, 1, 2)), (1, 0, 2, 3))
    cg = lm.compile(g, mem.hip)

    def call(seed):
        values = {t.id: normal(t.shape, seed + t.id) for t in (x, w, b)}
        mem.calls.clear()
        return values, cg(values)

    values, res = call(1)
    assert mem.calls == ["matmul 1", "map"]
    for walk in (list, tuple, lambda r: r[:], lambda r: [*reversed(r)], lambda r: r.copy(), lambda r: [y for y in r]):
        buffers = walk(res)
        assert len(buffers) == len(g.nodes) and all(isinstance(y, lm.HipArray) for y in buffers)
        del buffers
        call(2)
        gc.collect()
        assert mem.calls == ["matmul 1", "map"]
    blocks = len(mem.blocks)
    held = list(res)[biased.id]  # one of them is kept: it is up to date in every later call, and what it reads as well
    for seed in (3, 4):
        values, _ = call(seed)
        close(held.to_host(), values[x.id] @ values[w.id].T + values[b.id])
    assert res[biased.id] is held
    del held
    again = res[biased.id]  # asked for by number: the graph's from now on
    values, _ = call(6)
    close(again.to_host(), values[x.id] @ values[w.id].T + values[b.id])
    close(res[product.id].to_host(), values[x.id] @ values[w.id].T)
    assert len(mem.blocks) > blocks
