"""The nodes around attention on the device: lmh_matmul, lmh_map and lmh_copy_many at the edges of their tiles, against
float64 numpy and the reference's CPU semantics (HostOp.compute); and what a compiled graph does with nodes that
disappeared into another node's launch."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def _low(lm):
    return lm.host.lowering


# one case per form of the kernel (64 x 64, 32 x 64 and 32 x 32 tiles), each with remainders in every direction; the heads
# split with rows that cross sequences inside a tile; operands that take the register path (K % 4, 16-bit types)
@pytest.mark.parametrize("B,S,K,N,heads,dtype,bias", [
    (1, 1, 4, 1, 0, "f32", False), (1, 33, 36, 65, 0, "f32", True), (1, 700, 132, 1024, 0, "f32", False),
    (2, 1100, 64, 2100, 0, "f32", True), (3, 37, 68, 120, 5, "f32", True), (5, 7, 128, 64, 2, "f16", False),
    (2, 129, 256, 320, 5, "bf16", True), (1, 50, 30, 70, 0, "f32", True), (1, 63, 2050, 33, 3, "f32", False),
])
def test_projection_matches_float64(lm, hip, oracle, B, S, K, N, heads, dtype, bias):
    x, w = oracle.gen_normal((B, S, K), 31000 + S), oracle.gen_normal((N, K), 31100 + N, 1.0 / np.sqrt(K))
    bv = oracle.gen_normal((N,), 31200)
    dx, dw, db = (lm.to_device(a, hip) for a in (x, w, bv))
    out = lm.HipArray((B, heads, S, N // heads) if heads else (B, S, N), dtype, hip)
    p = (lm.binding.MatmulParams * 1)()
    assert _low(lm).fill_matmul(p[0], out, dx, dw, transposed=True, bias=db if bias else None, heads=heads)
    lm.binding.matmul(p, 1)
    want = x.astype(np.float64) @ w.astype(np.float64).T + (bv if bias else 0)
    if heads:
        want = np.transpose(np.reshape(want, (B, S, heads, N // heads), order="F"), (0, 2, 1, 3))
    assert rel_err(out.to_host(), want) <= {"f32": 2e-6, "f16": 5e-4, "bf16": 4e-3}[dtype]


# Large products of fp32 operands run on bf16 pieces: every tile (64 x 128, 64 x 64, 32 x 64) with remainders in every direction,
# heads whose rows cross sequences, 16-bit results. Against float64 with the bound of the fp32 product (its error is smaller).
@pytest.mark.parametrize("B,S,K,N,heads,dtype,bias", [
    (1, 701, 2052, 2500, 0, "f32", True), (2, 350, 2048, 2560, 20, "bf16", False), (1, 590, 580, 1150, 0, "f32", True),
    (3, 197, 576, 1152, 9, "f16", True), (1, 33, 772, 5000, 0, "f32", False), (1, 31, 1540, 9000, 10, "f32", True),
])
def test_products_on_pieces_match_float64(lm, hip, oracle, B, S, K, N, heads, dtype, bias):
    test_projection_matches_float64(lm, hip, oracle, B, S, K, N, heads, dtype, bias)


# ... and the tiles of 96 columns: 64 x 96 and 96 x 96
@pytest.mark.parametrize("B,S,K,N,heads,dtype,bias", [(1, 701, 2052, 2000, 0, "f32", True), (2, 351, 2048, 1940, 20, "bf16", False), (3, 458, 1540, 1530, 9, "f16", True), (1, 1390, 1028, 1450, 0, "f32", False)])
def test_products_on_pieces_of_96_columns(lm, hip, oracle, B, S, K, N, heads, dtype, bias):
    test_projection_matches_float64(lm, hip, oracle, B, S, K, N, heads, dtype, bias)
    if not heads:
        test_values_that_pieces_do_not_hold(lm, hip, oracle, S, K, N)


def test_products_of_rows_far_apart(lm, hip, oracle):
    """96 rows so far apart that the last one's byte offset takes more than 31 bits (64 rows' does not), beside a remainder of K."""
    M, K, N, step = 96, 1540, 24576, 5_800_000
    x, w = oracle.gen_normal((M, K), 37000), oracle.gen_normal((N, K), 37100)
    spread = np.ones(((M - 1) * step + K,), np.float32)
    for m in range(M):
        spread[m * step:m * step + K] = x[m]
    dx, dw, out = lm.to_device(spread, hip), lm.to_device(w, hip), lm.HipArray((1, M, N), "f32", hip)
    p = (lm.binding.MatmulParams * 1)()
    assert _low(lm).fill_matmul(p[0], out, lm.HipArray((1, M, K), "f32", hip), dw, transposed=True)
    p[0].a, p[0].a_stride[1] = dx.ptr, step
    lm.binding.matmul(p, 1)
    got = out.to_host()[0]
    # fp32 sums of K products, each within K 2^-24 of the sum of their magnitudes
    want, top = x.astype(np.float64) @ w.astype(np.float64).T, np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert (np.abs(got - want) <= K * 2.0 ** -24 * top).all()


@pytest.mark.parametrize("M,K,N", [(590, 580, 1150), (33, 772, 5000), (701, 2052, 2500)])
def test_values_that_pieces_do_not_hold(lm, hip, oracle, M, K, N):
    """Infinities, NaN, values next to the largest and rows far below the smallest normal bf16 piece: what fp32 gives."""
    x, w = oracle.gen_normal((M, K), 36000 + M), oracle.gen_normal((N, K), 36100 + N)
    x[0, 3], x[1, 5], x[2, 7], x[3, 9], w[4, 11] = np.inf, np.nan, -np.inf, 3.4e38, np.inf
    w[:, 9] *= 0.01
    x[:, 11] = np.where(np.arange(M) % 7 == 0, 0, x[:, 11])  # infinity times zero
    x[10:13] *= np.float32(2.0 ** -122)
    w[20:23] *= np.float32(2.0 ** -100)
    x[14] *= np.float32(2.0 ** 110)
    out = lm.HipArray((1, M, N), "f32", hip)
    p = (lm.binding.MatmulParams * 1)()
    dx, dw = lm.to_device(x[None], hip), lm.to_device(w, hip)
    assert _low(lm).fill_matmul(p[0], out, dx, dw, transposed=True)
    lm.binding.matmul(p, 1)
    got = out.to_host()[0]
    with np.errstate(all="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64).T
        top = np.abs(np.where(np.isfinite(x), x, 0)).astype(np.float64) @ np.abs(np.where(np.isfinite(w), w, 0)).astype(np.float64).T
    finite = np.abs(want) < 3e38
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    # fp32 sums of K products, each within K 2^-24 of the sum of their magnitudes (and within the smallest subnormal)
    assert (np.abs(got[finite] - want[finite]) <= K * 2.0 ** -24 * top[finite] + K * 2.0 ** -149).all()
    # rows of one magnitude each, as exact as any other row
    for rows in (slice(10, 13), slice(14, 15)):
        ok = np.r_[0:4, 5:20, 23:N]
        g, v = got[rows][:, ok].astype(np.float64), want[rows][:, ok]
        assert np.linalg.norm(g - v) <= 2e-6 * np.linalg.norm(v)


@pytest.mark.parametrize("a_shape,b_shape,dtypes", [
    ((3, 40, 72), (3, 72, 50), ("f32", "f32")), ((40, 72), (5, 72, 64), ("f32", "f16")), ((2, 3, 33, 20), (20, 100), ("bf16", "f32")),
])
def test_batched_products_of_any_type(lm, hip, oracle, a_shape, b_shape, dtypes):
    a, b = (oracle.round_to(oracle.gen_normal(s, 31300 + i), d) for i, (s, d) in enumerate(zip((a_shape, b_shape), dtypes)))
    got = lm.execute_op(lm.MatMulOp(), lm.to_device(a, hip, dtypes[0]), lm.to_device(b, hip, dtypes[1])).to_host()
    assert rel_err(got, np.matmul(a.astype(np.float64), b.astype(np.float64))) <= 2e-6


@pytest.mark.parametrize("shape,ops", [
    ((5,), [("expand", 0, 3)]), ((2, 70, 130), [("permute", 0, 2, 1)]), ((3, 65, 8, 9), [("permute", 0, 2, 1, 3), ("reshape", 3, 8, 585)]),
    ((2, 6, 40), [("reshape", 2, 6, 8, 5), ("permute", 0, 2, 1, 3), ("permute", 0, 2, 1, 3), ("reshape", 2, 6, 40)]),
    ((7, 11), [("reshape", 11, 7)]), ((1, 1, 64), [("permute", 2, 0, 1), ("expand", 3, 64)]),
])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_chains_of_moved_elements(lm, hip, oracle, shape, ops, dtype):
    g = lm.Graph()
    x = lm.tensor(g, shape, dtype)
    a = oracle.round_to(oracle.gen_normal(shape, 31400), dtype)
    node, want = x, a
    for kind, *args in ops:
        node = {"permute": lambda: lm.permute(node, args), "reshape": lambda: lm.reshape(node, args), "expand": lambda: lm.expand(node, *args)}[kind]()
        want = g.nodes[node.id].op.compute(want)
    np.testing.assert_array_equal(lm.execute(g, node.id, {x.id: a}, hip), want)
    b = oracle.gen_normal(want.shape[-1:], 31401)
    got = lm.execute_op(lm.AddOp(), lm.to_device(want, hip), lm.to_device(b, hip)).to_host()
    np.testing.assert_array_equal(got, want + b)


@pytest.mark.parametrize("offset", [0, 4])
def test_copies_of_every_length_in_one_launch(lm, hip, offset):
    lengths = [1, 15, 16, 17, 16383, 16384, 16385, 40000, 3, 100]  # more than one launch's worth
    rng = np.random.default_rng(5)
    src = [rng.integers(0, 1 << 30, n + 8, dtype=np.int32) for n in lengths]
    dev = [lm.to_device(s, hip) for s in src]
    out = [lm.to_device(np.full(n + 8, -1, np.int32), hip) for n in lengths]
    copies = _low(lm).CopyList([(o.ptr + offset, d.ptr + offset, n * 4 - (1 if n > 1 else 0)) for o, d, n in zip(out, dev, lengths)])
    copies.launch()
    for s, o, n in zip(src, out, lengths):
        got, nbytes = o.to_host().view(np.uint8), n * 4 - (1 if n > 1 else 0)
        want = np.full((n + 8) * 4, 255, np.uint8)
        want[offset:offset + nbytes] = s.view(np.uint8)[offset:offset + nbytes]
        np.testing.assert_array_equal(got, want)


def test_a_node_inside_a_launch_is_computed_once_it_is_asked_for(lm, hip, oracle):
    B, S, hidden, heads = 2, 20, 64, 4
    g = lm.Graph()
    x = lm.tensor(g, (B, S, hidden))
    layer = lm.SelfAttention(hidden, heads, heads, g)
    out = layer(x)
    product = next(i for i, n in enumerate(g.nodes) if isinstance(n.op, lm.MatMulOp))
    cg = lm.compile(g, hip)
    ws = {p.weight.id: oracle.gen_normal((hidden, hidden), 31500 + i, 0.1) for i, p in
          enumerate((layer.q_proj, layer.k_proj, layer.v_proj, layer.o_proj))}
    first = cg({x.id: oracle.gen_normal((B, S, hidden), 31600), **ws})[out.id].to_host()
    buffer = cg.results[product]  # handed out: kept up to date from here on
    for seed in (31601, 31602):
        xs = oracle.gen_normal((B, S, hidden), seed)
        res = cg({x.id: lm.to_device(xs, hip)})
        want = xs.astype(np.float64) @ ws[layer.q_proj.weight.id].astype(np.float64).T
        assert rel_err(buffer.to_host(), want) <= 2e-6 and res[product] is buffer
        np.testing.assert_array_equal(res[out.id].to_host(), lm.execute(g, out.id, {x.id: xs, **ws}, hip))
    np.testing.assert_array_equal(cg({x.id: oracle.gen_normal((B, S, hidden), 31600)})[out.id].to_host(), first)


def test_inputs_that_overlap_are_copied_in_their_order(lm, hip, oracle):
    g = lm.Graph()
    a, b = lm.tensor(g, (64,)), lm.tensor(g, (64,))
    out = lm.add(a, b)
    cg = lm.compile(g, hip)
    va, vb = oracle.gen_normal((64,), 1), oracle.gen_normal((64,), 2)
    cg({a.id: va, b.id: vb})
    res = cg({a.id: cg.results[b.id], b.id: cg.results[a.id]})  # a takes b's values, then b takes a's new ones
    np.testing.assert_array_equal(res[out.id].to_host(), vb + vb)


def test_copies_that_meet_keep_their_order(lm, hip):
    rng = np.random.default_rng(6)
    n = 30000
    host = rng.integers(0, 1 << 30, 8 * n, dtype=np.int32)
    for _ in range(20):
        dev, want = lm.to_device(host, hip), host.copy()
        ranges = []
        for _ in range(int(rng.integers(2, 20))):
            length = int(rng.integers(0, n))
            dst, src = (int(x) for x in rng.integers(0, 8 * n - length, 2))
            if abs(dst - src) < length:  # (a range that meets itself is the runtime's copy, whose order is its own)
                dst = src
            ranges.append((dst, src, length))
            want[dst:dst + length] = want[src:src + length].copy()
        _low(lm).CopyList([(dev.ptr + 4 * d, dev.ptr + 4 * s, 4 * k) for d, s, k in ranges]).launch()
        np.testing.assert_array_equal(dev.to_host(), want)


@pytest.mark.parametrize("M,K,N", [(701, 2048, 2000), (590, 580, 1150), (33, 772, 5000), (1390, 1028, 1450), (100, 768, 768), (5, 33, 70), (1400, 2052, 2500)])
def test_products_of_operands_in_the_callers_arrays(lm, hip, oracle, M, K, N):
    """A compiled graph that begins with a product leaves the same memory behind whether its inputs are copied in front of it or
    read where they lie; also with an input one element off 16 bytes, the weight fed as well, and the result fed back."""
    g = lm.Graph()
    x, w, other = lm.tensor(g, (1, M, K)), lm.tensor(g, (K, N)), lm.tensor(g, (3, 4099))
    out = lm.matmul(x, w)
    fed, plain = lm.compile(g, hip), lm.compile(g, hip)
    assert fed._fed is not None
    plain._fed = None
    rng = np.random.default_rng(M)

    def array(shape, skip=0):
        whole = lm.to_device(rng.standard_normal(int(np.prod(shape)) + skip).astype(np.float32), hip)
        part = whole.view(whole.shape)
        part.shape, part.nbytes, part.ptr = shape, whole.nbytes - 4 * skip, whole.ptr + 4 * skip
        return part

    def back(cg):  # the front of the graph's own result
        v = cg.results[out.id].view((1, M, N))
        v.shape, v.nbytes = (3, 4099), 4 * 3 * 4099
        return v

    for feeds in ({x.id: array((1, M, K)), w.id: array((K, N)), other.id: array((3, 4099))}, {x.id: array((1, M, K))},
                  {x.id: array((1, M, K), 1), other.id: array((3, 4099), 2)}, {other.id: back, x.id: array((1, M, K))}):
        if M * N < 3 * 4099 and other.id in feeds and callable(feeds[other.id]):
            continue
        for cg in (fed, plain):
            cg({k: v(cg) if callable(v) else v for k, v in feeds.items()})
        lm.binding.sync()
        for t in (x, w, other, out):
            np.testing.assert_array_equal(fed.results[t.id].to_host(), plain.results[t.id].to_host())
        assert np.abs(fed.results[out.id].to_host()).max() > 0


@pytest.mark.parametrize("M,K,N", [(590, 580, 1150), (33, 772, 5000), (701, 2052, 2500), (701, 2052, 2000), (1390, 1028, 1450)])
def test_a_product_left_to_a_small_element(lm, hip, oracle, M, K, N):
    """One element of a row far below the others of it, and the only one that meets something: its product with all its bits, on
    every tile that takes bf16 pieces."""
    x, w = oracle.gen_normal((M, K), 38000 + M), oracle.gen_normal((N, K), 38100 + N)
    small = [2.0 ** -e for e in (100, 104, 108, 112, 116, 120, 124)]
    # the column where the rows meet; large values of x's and of w's row in front of it that meet zeros (64 columns apart: a lane
    # of the kernel reads them all)
    k, at_x, at_w = 64 * 5 + 9, slice(72, 77), slice(136, 141)
    x[:, k], w[:, k] = 1 + np.abs(x[:, k]), 1 + np.abs(w[:, k])
    x[:, at_w], w[:, at_x] = 0, 0
    for i, e in enumerate(small):
        x[3 * i], x[3 * i, at_x], x[3 * i, k] = 0, 1.5, 1.2345678 * e
        w[40 + i], w[40 + i, at_w], w[40 + i, k] = 0, 1.5, -1.1234567 * e
    out = lm.HipArray((1, M, N), "f32", hip)
    p = (lm.binding.MatmulParams * 1)()
    dx, dw = lm.to_device(x[None], hip), lm.to_device(w, hip)
    assert _low(lm).fill_matmul(p[0], out, dx, dw, transposed=True)
    lm.binding.matmul(p, 1)
    got = out.to_host()[0].astype(np.float64)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    others = np.r_[0:40, 47:N]
    for i in range(len(small)):  # one product each: its rounding, and that of the pieces left out
        a, b = got[3 * i, others], want[3 * i, others]
        assert (np.abs(a - b) <= 2.0 ** -22 * np.abs(b)).all(), small[i]
        a, b = got[21:, 40 + i], want[21:, 40 + i]
        assert (np.abs(a - b) <= 2.0 ** -22 * np.abs(b)).all(), small[i]


@pytest.mark.parametrize("M,K,N,dtype", [(700, 2048, 2560, "f32"), (701, 2052, 2000, "bf16"), (590, 580, 1156, "f16")])
def test_products_on_pieces_into_results_of_any_alignment(lm, hip, oracle, M, K, N, dtype):
    """Results that begin between 16-byte addresses are stored column by column: the bits of the aligned ones, nothing beside them."""
    x, w, bv = oracle.gen_normal((1, M, K), 38000), oracle.gen_normal((N, K), 38100, 1.0 / np.sqrt(K)), oracle.gen_normal((N,), 38200)
    dx, dw, db = (lm.to_device(a, hip) for a in (x, w, bv))
    out, wide = lm.HipArray((1, M, N), dtype, hip), lm.HipArray((M * N + 8,), dtype, hip).fill_bytes(0xff)
    p = (lm.binding.MatmulParams * 1)()
    assert _low(lm).fill_matmul(p[0], out, dx, dw, transposed=True, bias=db)
    lm.binding.matmul(p, 1)
    esz = 4 if dtype == "f32" else 2
    p[0].c = wide.ptr + 3 * esz
    lm.binding.matmul(p, 1)
    got = wide.to_host()
    np.testing.assert_array_equal(got[3:3 + M * N].reshape(1, M, N), out.to_host())
    assert np.isnan(got[:3]).all() and np.isnan(got[3 + M * N:]).all()  # (0xffff is a NaN in every type)
    assert rel_err(out.to_host(), x.astype(np.float64) @ w.astype(np.float64).T + bv) <= {"f32": 2e-6, "f16": 5e-4, "bf16": 4e-3}[dtype]
