"""Sequences of a block's dispatches that run as fewer kernels (copy + RMS norm + the split before Q8_0 products; product +
bias + residual): every buffer holds bit for bit what it holds when each dispatch is a kernel of its own."""
import functools

import numpy as np
import pytest

from loadngo_amd import compute as C
from tests.gpu_common import gpu  # noqa: F401
from tests.helpers import from_bf16_bits, q8_test_matrix, to_bf16_bits, xorshift_values

pytestmark = pytest.mark.gpu
_matrix = functools.lru_cache(maxsize=None)(q8_test_matrix)


def both_ways(gpu, arrays, record):
    """Every buffer after `record` ran on fresh copies of the arrays, fused and not."""
    out = []
    try:
        for fusing in (True, False):
            gpu.debug_set("LNG_NO_FUSING", None if fusing else "1")
            bufs = [gpu.upload(a) for a in arrays]
            batch = gpu.batch(bufs)
            record(batch)
            done = batch.run()
            assert not isinstance(done.gpu_time, Exception), done.gpu_time
            batch.drop()
            out.append([b.read(np.uint8) for b in bufs])
            for b in bufs:
                b.free()
    finally:
        gpu.debug_set("LNG_NO_FUSING", None)
    return out


@pytest.mark.parametrize("n,cols,src_stride,x_stride,offset", [
    (1, 2880, 2880, 2880, 0), (31, 2880, 2880, 2880, 0), (33, 2880, 2880, 2880, 0), (77, 288, 292, 288, 0), (64, 4096, 4096, 4100, 0),
    (64, 4128, 4128, 4128, 0), (64, 256, 256, 256, 0), (100, 288, 288, 288, 4), (1281, 288, 288, 288, 0), (1300, 320, 320, 324, 0)])
def test_copy_norm_and_split_in_one_kernel(gpu, n, cols, src_stride, x_stride, offset):
    """Positions up to and past both ways of splitting, row widths at the edges of the norm kernels, strides, hidden rows
    off a 16-byte boundary; one product and three, a product of other rows in between, the norm alone."""
    eps, rows = 1e-5, 80
    mats = [q8_test_matrix(rows, cols, 30 + i) for i in range(3)]
    h = 3 * xorshift_values(71 + n, n * src_stride + 1)
    x = xorshift_values(72, n * x_stride)
    weights = 1 + 0.2 * xorshift_values(73, cols)
    arrays = [h, x, weights, np.zeros(6 * n * rows, np.float32)]
    for codes, bits, _ in mats:
        arrays += [codes, bits]
    hs = C.Slice(0, offset, ((n - 1) * src_stride + cols) * 4)
    xs, ws = C.Slice(1, 0, ((n - 1) * x_stride + cols) * 4), C.Slice(2, 0, cols * 4)
    matrix = lambda i: (C.Slice(4 + 2 * i, 0, rows * cols), C.Slice(5 + 2 * i, 0, rows * cols // 16))  # noqa: E731
    y = lambda i: C.Slice(3, i * n * rows * 4, n * rows * 4)  # noqa: E731

    def record(batch):
        batch.copy_rows((hs, src_stride), (xs, x_stride), n, cols)
        batch.rmsnorm_rows((xs, ws), n, (cols, x_stride), eps)
        batch.gemm_q8_0_many([(matrix(i), y(i), rows) for i in range(3)], xs, cols, n, x_stride)
        batch.rmsnorm_rows((xs, ws), n, (cols, x_stride), eps)                           # without a copy
        batch.gemm_q8_0(matrix(0), xs, y(3), rows, cols, n, (x_stride, rows))
        batch.copy_rows((hs, src_stride), (xs, x_stride), n, cols)                       # without a norm
        batch.gemm_q8_0(matrix(1), xs, y(4), rows, cols, n, (x_stride, rows))
        if n > 1:                                                                        # the norm of fewer rows than are copied
            batch.copy_rows((hs, src_stride), (xs, x_stride), n, cols)
            batch.rmsnorm_rows((C.Slice(1, 0, ((n - 2) * x_stride + cols) * 4), ws), n - 1, (cols, x_stride), eps)
            batch.gemm_q8_0(matrix(2), xs, y(5), rows, cols, n, (x_stride, rows))

    fused, apart = both_ways(gpu, arrays, record)
    for i, (a, b) in enumerate(zip(fused, apart)):
        assert np.array_equal(a, b), "buffer %d" % i
    got = fused[3].view(np.float32).reshape(6, n, rows)
    hidden = np.stack([h[offset // 4 + p * src_stride:][:cols] for p in range(n)]).astype(np.float64)
    once = hidden / np.sqrt((hidden * hidden).mean(axis=1, keepdims=True) + eps) * weights
    twice = once / np.sqrt((once * once).mean(axis=1, keepdims=True) + eps) * weights
    for y_i, positions, i in ((0, once, 0), (1, once, 1), (2, once, 2), (3, twice, 0), (4, hidden, 1)):
        want = positions @ mats[i][2].T
        assert np.abs(got[y_i] - want).max() / np.abs(want).max() < 1e-5, y_i  # the reference's bound (glue.rs:171)


@pytest.mark.parametrize("d,stride", [(264, 264), (1024, 1028), (1032, 1032), (4088, 4092), (4096, 4096)])
def test_norm_at_the_edges_of_its_words(gpu, d, stride):
    """Rows that end within a thread's share of words, and gaps between rows that stay as they are."""
    rows, eps = 5, 1e-5
    x, w = 3 * xorshift_values(91, (rows - 1) * stride + d), 1 + 0.2 * xorshift_values(92, d)
    bufs = [gpu.upload(x), gpu.upload(w)]
    batch = gpu.batch(bufs)
    batch.rmsnorm_rows((C.Slice(0, 0, x.nbytes), C.Slice(1, 0, w.nbytes)), rows, (d, stride), eps)
    done = batch.run()
    assert not isinstance(done.gpu_time, Exception), done.gpu_time
    got = bufs[0].read(np.float32)
    batch.drop()
    for b in bufs:
        b.free()
    for r in range(rows):
        row = x[r * stride:r * stride + d].astype(np.float64)
        want = row / np.sqrt((row * row).mean() + eps) * w
        assert np.abs(got[r * stride:r * stride + d] - want).max() <= 1e-6 * np.abs(want).max()  # (a sum of 4,096 squares and three roundings in f32)
        assert np.array_equal(got[r * stride + d:(r + 1) * stride], x[r * stride + d:(r + 1) * stride])


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("n,rows,cols", [(1, 48, 96), (7, 33, 64), (17, 48, 96), (32, 64, 96), (77, 100, 64), (200, 192, 96), (1290, 260, 64),
                                         (2, 4112, 2048), (16, 5121, 2912), (1, 8201, 96)])
def test_bias_and_residual_in_the_product(gpu, n, rows, cols, bf16):
    """Each kind of product with bias and residual, bias or residual alone, and the sequences that only look alike: hidden
    rows over the positions, over the codes or over the bias, a residual of another width, the bias added twice, y with gaps,
    a second residual."""
    codes, bits, _ = q8_test_matrix(rows, cols, 51)
    x = xorshift_values(52 + n, n * cols)
    x = to_bf16_bits(x) if bf16 else x
    room = np.zeros(max(n * rows * 4, 4096) // 4 * 4, np.uint8)
    x_held, codes_held = np.concatenate([x.view(np.uint8), room]), np.concatenate([codes.view(np.uint8), room])
    bias_held = xorshift_values(53, n * rows)  # the bias is its first row
    arrays = [x_held, codes_held, bits, bias_held, xorshift_values(54, n * rows), np.zeros(8 * n * rows, np.float32), np.zeros(n * (rows + 4), np.float32)]
    es = 2 if bf16 else 4
    xs, m = C.Slice(0, 0, n * cols * es), (C.Slice(1, 0, rows * cols), C.Slice(2, 0, rows * cols // 16))
    bs, hs, size = C.Slice(3, 0, rows * 4), C.Slice(4, 0, n * rows * 4), n * rows * 4

    def product(batch, y, stride=rows):
        (batch.gemm_q8_0_bf16 if bf16 else batch.gemm_q8_0)(m, xs, y, rows, cols, n, (cols, stride))

    def record(batch):
        y = [C.Slice(5, i * size, size) for i in range(8)]
        product(batch, y[0])
        batch.add_rows(y[0], (bs, 0), n, rows)
        batch.add_rows(hs, (y[0], rows), n, rows)
        product(batch, y[1])
        batch.add_rows(y[1], (bs, 0), n, rows)                                   # the bias alone, then twice
        batch.add_rows(y[1], (bs, 0), n, rows)
        product(batch, y[2])
        batch.add_rows(hs, (y[2], rows), n, rows)                                # the residual alone, then twice, then the bias
        batch.add_rows(hs, (y[2], rows), n, rows)
        batch.add_rows(y[2], (bs, 0), n, rows)
        product(batch, y[3])
        batch.add_rows(y[3], (C.Slice(3, 0, size), rows), n, rows)               # another row for every position
        batch.add_rows(y[4], (y[3], rows), n, rows)                              # and a residual that is no hidden state
        strided = C.Slice(6, 0, ((n - 1) * (rows + 4) + rows) * 4)
        product(batch, strided, rows + 4)
        batch.add_rows(hs, (strided, rows + 4), n, rows)                         # y with gaps
        product(batch, y[5])
        batch.add_rows(y[5], (bs, 0), n, rows)
        batch.add_rows(C.Slice(3, 0, size), (y[5], rows), n, rows)               # over the bias
        product(batch, y[6])
        batch.add_rows(C.Slice(1, 0, size), (y[6], rows), n, rows)               # over the codes
        product(batch, y[7])
        batch.add_rows(C.Slice(0, 0, size), (y[7], rows), n, rows)               # over the positions
        product(batch, y[7])

    fused, apart = both_ways(gpu, arrays, record)
    for i, (a, b) in enumerate(zip(fused, apart)):
        assert np.array_equal(a, b), "buffer %d" % i
    assert not np.isnan(fused[5].view(np.float32)[:6 * n * rows]).any()


@pytest.mark.parametrize("dtype", [C.F32, C.BF16])
@pytest.mark.parametrize("n,one_item,dim,rotary,bias,normed,kind,cols,heads,kv_heads", [(*c, 96, 6, 2) for c in (
    (1, True, 64, 64, True, True, ""), (1, True, 64, 64, False, False, ""), (2, False, 64, 64, True, True, ""), (16, False, 64, 64, True, True, ""),
    (3, True, 64, 64, True, False, ""), (16, True, 64, 64, False, True, ""), (17, False, 64, 64, True, True, ""), (5, False, 64, 32, True, True, ""),
    (2, False, 128, 128, True, True, ""), (4, False, 64, 64, True, True, "backwards"), (4, False, 64, 64, True, True, "swapped"),
    (4, False, 64, 64, True, True, "table over q"), (4, False, 64, 64, True, True, "queries over x"))] + [
    (1, True, 64, 64, True, True, "", 2880, 6, 2), (16, False, 64, 64, True, True, "", 2880, 6, 2), (5, False, 64, 64, True, False, "", 2880, 6, 2),
    (1, True, 64, 64, True, True, "", 352, 64, 8), (16, True, 64, 64, False, False, "", 352, 64, 8), (1, True, 64, 64, False, False, "", 4160, 2, 1),
    (7, False, 64, 64, True, False, "", 4160, 2, 1), (1, True, 64, 64, True, True, "", 12288, 2, 1), (3, False, 64, 64, True, True, "", 12288, 2, 1),
    (6, False, 64, 64, True, False, "", 16416, 2, 1), (9, False, 64, 64, True, True, "", 512, 6, 2), (16, False, 64, 64, True, False, "", 544, 6, 2),
    # more rows than a workgroup of 16 a unit takes: tiles of 18 to 32 rows, across heads
    (2, False, 64, 64, True, True, "", 2880, 64, 8), (5, True, 64, 64, True, True, "", 2880, 64, 8), (16, False, 64, 64, False, True, "", 2880, 64, 8),
    (16, True, 64, 64, True, False, "", 2912, 56, 7), (2, False, 64, 64, False, False, "", 4096, 64, 8), (5, False, 64, 64, True, True, "", 4064, 66, 11),
    (16, False, 64, 64, True, True, "", 4096, 96, 16), (9, True, 64, 64, True, True, "", 2048, 66, 1), (1, True, 64, 64, True, True, "", 96, 112, 16)])
def test_projections_and_preparation_in_one_kernel(gpu, n, one_item, dim, rotary, bias, normed, kind, cols, heads, kv_heads, dtype):
    """q, k and v of up to 16 positions with the preparation after them: tables of items and one item, rings that wrap, with
    and without biases and norm; and what stays apart: more positions, other widths, items in another order than the rows, k
    and v the other way round, a rotation table in rows that q is written to, prepared queries where x is. Columns: fewer
    pairs of blocks than wavefronts, several pairs a wavefront, more than one turn of 4,096, a block left over, scales that
    wait in LDS in more than 64 words a row or do not fit there; positions split by the product itself, in tiles of 16 rows and of more,
    and before it. The products and the prepared rows against float64, too."""
    slots, eps = 24, 1e-5
    qw, kw, es = heads * dim, kv_heads * dim, 4 if dtype == C.F32 else 2
    elements = []
    mats = []
    for i, rows in enumerate((qw, kw, kw)):
        codes, bits, e = _matrix(rows, cols, 60 + i)
        mats.append((codes, bits))
        elements.append(e)
    arrays = [3 * xorshift_values(81 + n, n * max(cols, qw)), 1 + 0.2 * xorshift_values(82, cols), xorshift_values(83, n * qw),
              np.zeros(2 * n * kw, np.float32), xorshift_values(84, n * rotary), np.zeros(n * qw * es, np.uint8),
              np.zeros(2 * n * slots * kw * es, np.uint8), xorshift_values(85, qw + 2 * kw)]
    for codes, bits in mats:
        arrays += [codes, bits]
    table, q_out = (2 if kind == "table over q" else 4), (0 if kind == "queries over x" else 5)
    k_at, v_at = (n * kw * 4, 0) if kind == "swapped" else (0, n * kw * 4)
    order = list(range(n))[::-1] if kind == "backwards" else list(range(n))
    item = lambda i, j, rows, start: C.PrepareItem(  # noqa: E731
        q_offset=j * qw * 4, k_offset=j * kw * 4, v_offset=n * kw * 4 + j * kw * 4, table_offset=j * rotary * 4, q_out_offset=j * qw * es,
        k_cache_offset=i * slots * kw * es, v_cache_offset=(n + i) * slots * kw * es, n=rows, start=start, slots=slots)
    items = C.prepare_items([item(0, 0, n, slots - 1)] if one_item else [item(i, j, 1, 5 + 13 * i) for i, j in enumerate(order)])
    biases = [C.Slice(7, 0, qw * 4), C.Slice(7, qw * 4, kw * 4), C.Slice(7, (qw + kw) * 4, kw * 4)] if bias else [None] * 3

    def record(batch):
        many = [((C.Slice(8 + 2 * i, 0, rows * cols), C.Slice(9 + 2 * i, 0, rows * cols // 16)), y, rows)
                for i, (rows, y) in enumerate(((qw, C.Slice(2, 0, n * qw * 4)), (kw, C.Slice(3, k_at, n * kw * 4)), (kw, C.Slice(3, v_at, n * kw * 4))))]
        xs = C.Slice(0, 0, n * cols * 4)
        if normed:
            batch.gemm_q8_0_many_normed(many, xs, (C.Slice(1, 0, cols * 4), eps), cols, n, cols)
        else:
            batch.gemm_q8_0_many(many, xs, cols, n, cols)
        batch.prepare_attention(dict(q=2, k=3, v=3, table=table, q_out=q_out, k_cache=6, v_cache=6), items, heads, kv_heads, dim, rotary, dtype, *biases)

    fused, apart = both_ways(gpu, arrays, record)
    for i, (a, b) in enumerate(zip(fused, apart)):
        assert np.array_equal(a, b), "buffer %d" % i
    assert fused[5 if q_out == 5 else 0].any() and fused[6].any()
    if kind or rotary != 64 or dim != 64:
        return
    x = arrays[0][:n * cols].reshape(n, cols).astype(np.float64)
    if normed:
        x = x / np.sqrt((x * x).mean(axis=1, keepdims=True) + eps) * arrays[1]
    want = [x @ e.T for e in elements]
    tol = [1e-5 * np.abs(w).max() for w in want]  # the reference's bound of the products (glue.rs:171)
    got_kv = fused[3].view(np.float32).reshape(2, n, kw)
    for got, w, t in zip((fused[2].view(np.float32)[:n * qw].reshape(n, qw), got_kv[0], got_kv[1]), want, tol):
        assert np.abs(got - w).max() <= t
    if bias:
        want = [w + b for w, b in zip(want, np.split(arrays[7].astype(np.float64), [qw, qw + kw]))]
    angles = arrays[4][:n * 64].reshape(n, 1, 32, 2).astype(np.float64)  # cosine and sine of every pair

    def rotate(rows):
        r = rows.reshape(n, -1, 2, 32)
        low, high = r[:, :, 0], r[:, :, 1]
        return np.stack([low * angles[..., 0] - high * angles[..., 1], high * angles[..., 0] + low * angles[..., 1]], axis=2).reshape(n, -1)

    want = [rotate(want[0]), rotate(want[1]), want[2]]
    values = (lambda raw: raw.view(np.float32)) if dtype == C.F32 else (lambda raw: from_bf16_bits(raw.view(np.uint16)))
    caches = values(fused[6]).reshape(2, n, slots, kw)
    at = [(0, (slots - 1 + p) % slots) if one_item else (p, (5 + 13 * p) % slots) for p in range(n)]
    got = [values(fused[5]).reshape(n, qw), np.stack([caches[0][c, s] for c, s in at]), np.stack([caches[1][c, s] for c, s in at])]
    for g, w, t in zip(got, want, tol):  # a rotated value is two products of values that far off, each times at most 1.2; narrowing: half of 2^-8
        assert (np.abs(g - w) <= 3 * t + 1e-6 + (0 if dtype == C.F32 else 2.0 ** -8) * np.abs(w)).all()
