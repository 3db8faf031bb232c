"""GPU parity of the Q8_0 products (Batch::gemv_q8_0 / gemm_q8_0 / gemm_q8_0_tiled) through the C
ABI: the reference's own test (metal-compute/tests/q8_0_and_gpt_oss_glue.rs:155-177: its matrices,
shapes and bound, largest error below 1e-5 of the largest |y| against float64), strides, refusals,
and the tiny-model golden with the device doing projections, pre-attention step and attention."""
import os

import numpy as np
import pytest

from loadngo_amd import compute as C
from oracle import oracle as orc
from oracle import tiny_model as tm
from tests.gpu_common import gpu  # noqa: F401
from tests.helpers import REF_Q8_CASES, q8_test_matrix, xorshift_values
from tests.test_gpu_tiny_model import FIXTURE, TOLERANCE, DeviceSession

pytestmark = pytest.mark.gpu


def q8_run(gpu, codes, bits, x, rows, cols, kind, y_stride=None):
    n, x_stride = x.shape
    y_stride = rows if y_stride is None else y_stride
    y_len = ((n - 1) * y_stride + rows) * 4
    bufs = [gpu.upload(codes), gpu.upload(bits), gpu.upload(x), gpu.buffer(y_len)]
    bufs[3].fill(0xFF)
    batch = gpu.batch(bufs)
    m = (C.Slice(0, 0, codes.nbytes), C.Slice(1, 0, bits.nbytes))
    xs, ys = C.Slice(2, 0, ((n - 1) * x_stride + cols) * 4), C.Slice(3, 0, y_len)
    try:
        if kind == "gemv":
            batch.gemv_q8_0(m, xs, ys, rows, cols)
        elif kind == "gemm":
            batch.gemm_q8_0(m, xs, ys, rows, cols, n, (x_stride, y_stride))
        else:
            batch.gemm_q8_0_tiled(m, xs, ys, rows, cols, n, (x_stride, y_stride))
        assert batch.dispatches() == 1
        done = batch.run()
        assert not isinstance(done.gpu_time, Exception), done.gpu_time
        raw = bufs[3].read(np.float32)
    finally:
        batch.drop()
        for b in bufs:
            b.free()
    out = np.full((n, y_stride), np.nan, np.float32)
    out.reshape(-1)[:raw.size] = raw
    return out


@pytest.mark.parametrize("rows,cols,n,kind", REF_Q8_CASES + [(4096, 2880, 16, "gemm"), (2880, 4096, 31, "gemm"),
                                                             (5120, 2880, 512, "tiled"), (64, 32, 32, "tiled")])
def test_products_match_the_float64_definition(gpu, rows, cols, n, kind):
    codes, bits, elements = q8_test_matrix(rows, cols, 7 + rows)
    x = xorshift_values(11, n * cols).reshape(n, cols)
    want = x.astype(np.float64) @ elements.T
    got = q8_run(gpu, codes, bits, x, rows, cols, kind)
    assert not np.isnan(got).any()
    error = np.abs(got - want).max() / np.abs(want).max()
    assert error < 1e-5, f"{rows} x {cols}, {n} positions, {kind}: relative error {error:e}"  # glue.rs:171
    # and against the f32 CPU form, whose own distance from float64 is of the same size
    cpu = orc.q8_mul(codes, bits, x, rows, cols)
    assert np.abs(got - cpu).max() / np.abs(want).max() < 2e-5


@pytest.mark.parametrize("rows,cols,n,kind", [(320, 96, 1120, "tiled"), (2112, 64, 1056, "tiled"), (576, 160, 4224, "tiled"),
                                              (256, 32, 1024, "tiled"), (300, 96, 1100, "gemm"), (2100, 64, 1030, "gemm")])
def test_product_with_eight_position_tiles_or_more(gpu, rows, cols, n, kind):
    """From eight tiles of 128 positions on, workgroup ids are mapped to tiles per XCD in blocks of 8 row
    tiles x 4 position tiles and the grid is rounded up to whole blocks: every tile must be computed exactly
    once (ragged tile counts in both directions, ids without a tile), nothing outside y written."""
    codes, bits, elements = q8_test_matrix(rows, cols, 40 + rows)
    x = xorshift_values(13, n * cols).reshape(n, cols)
    want = x.astype(np.float64) @ elements.T
    got = q8_run(gpu, codes, bits, x, rows, cols, kind, y_stride=rows + 4)
    assert not np.isnan(got[:, :rows]).any()
    assert np.abs(got[:, :rows] - want).max() / np.abs(want).max() < 1e-5
    assert np.isnan(got[:-1, rows:]).all()           # 0xFF fill: gaps of y untouched


@pytest.mark.parametrize("rows,cols,n", [(4096, 2880, 1), (512, 2880, 5), (37, 96, 13), (2880, 4096, 32), (2880, 4096, 31),
                                         (320, 96, 1120), (2100, 64, 1030), (64, 32, 32), (5120, 2880, 512)])
def test_product_of_bf16_positions(gpu, rows, cols, n):
    """gemm_q8_0_bf16 (no counterpart in the reference): positions given in bf16, as a bf16 attention leaves them
    for the output projection. Against the float64 product of the same bf16 values, the reference's bound for
    its f32 kernels (glue.rs:171); strided x and y, gaps of y untouched."""
    from tests.helpers import from_bf16_bits, to_bf16_bits
    codes, bits, elements = q8_test_matrix(rows, cols, 60 + rows)
    x_stride, y_stride = cols + 8, rows + 4
    xb = np.full((n, x_stride), 0x7FC0, np.uint16)            # NaN between the rows of x: never read
    xb[:, :cols] = to_bf16_bits(xorshift_values(19, n * cols).reshape(n, cols))
    want = from_bf16_bits(xb[:, :cols]).astype(np.float64) @ elements.T
    y_len = ((n - 1) * y_stride + rows) * 4
    bufs = [gpu.upload(codes), gpu.upload(bits), gpu.upload(xb), gpu.buffer(y_len)]
    bufs[3].fill(0xFF)
    batch = gpu.batch(bufs)
    try:
        batch.gemm_q8_0_bf16((C.Slice(0, 0, codes.nbytes), C.Slice(1, 0, bits.nbytes)),
                             C.Slice(2, 0, ((n - 1) * x_stride + cols) * 2), C.Slice(3, 0, y_len), rows, cols, n,
                             (x_stride, y_stride))
        done = batch.run()
        assert not isinstance(done.gpu_time, Exception), done.gpu_time
        raw = bufs[3].read(np.float32)
    finally:
        batch.drop()
        for b in bufs:
            b.free()
    got = np.full((n, y_stride), np.nan, np.float32)
    got.reshape(-1)[:raw.size] = raw
    assert not np.isnan(got[:, :rows]).any()
    assert np.abs(got[:, :rows] - want).max() / np.abs(want).max() < 1e-5
    assert np.isnan(got[:-1, rows:]).all()


def test_strided_positions_and_untouched_gaps(gpu):
    rows, cols, n = 80, 96, 21
    codes, bits, elements = q8_test_matrix(rows, cols, 3)
    x = np.full((n, cols + 8), np.nan, np.float32)   # the gap between rows of x is never read
    x[:, :cols] = xorshift_values(5, n * cols).reshape(n, cols)
    got = q8_run(gpu, codes, bits, x, rows, cols, "gemm", y_stride=rows + 12)
    want = x[:, :cols].astype(np.float64) @ elements.T
    assert np.abs(got[:, :rows] - want).max() / np.abs(want).max() < 1e-5
    assert np.isnan(got[:-1, rows:]).all()           # 0xFF fill: gaps of y untouched


@pytest.mark.parametrize("n", [1, 9])
def test_scales_at_an_offset_of_two_bytes(gpu, n):
    """The reference asks 2-byte alignment of the scales (apple.rs:1799-1811); the few-position kernel copies
    a workgroup's scales to LDS a dword at a time only when they start on a 4-byte boundary."""
    rows, cols = 96, 160
    codes, bits, elements = q8_test_matrix(rows, cols, 21)
    x = xorshift_values(17, n * cols).reshape(n, cols)
    padded = np.concatenate([np.array([0x7E00], np.uint16), bits])   # a NaN in front of the scales
    bufs = [gpu.upload(codes), gpu.upload(padded), gpu.upload(x), gpu.buffer(n * rows * 4)]
    batch = gpu.batch(bufs)
    m = (C.Slice(0, 0, codes.nbytes), C.Slice(1, 2, bits.nbytes))
    try:
        if n == 1:
            batch.gemv_q8_0(m, C.Slice(2, 0, x.nbytes), C.Slice(3, 0, rows * 4), rows, cols)
        else:
            batch.gemm_q8_0(m, C.Slice(2, 0, x.nbytes), C.Slice(3, 0, n * rows * 4), rows, cols, n, (cols, rows))
        done = batch.run()
        assert not isinstance(done.gpu_time, Exception), done.gpu_time
        got = bufs[3].read(np.float32).reshape(n, rows)
    finally:
        batch.drop()
        for b in bufs:
            b.free()
    want = x.astype(np.float64) @ elements.T
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-5


def test_refusals_of_the_reference(gpu):
    """q8_0_and_gpt_oss_glue.rs:180-210 and the checks of apple.rs:889-894, 995-999, 1799-1806, 1868-1872."""
    bufs = [gpu.buffer(1 << 16) for _ in range(4)]
    res = gpu.resident(np.zeros(1 << 14, np.float32))
    batch = gpu.batch(bufs)
    s = lambda b, n: C.Slice(b, 0, n)
    with pytest.raises(C.Dispatch):   # rows of 40 are not whole blocks
        batch.gemv_q8_0((s(0, 160), s(1, 10)), s(2, 160), s(3, 16), 4, 40)
    with pytest.raises(C.Dispatch):   # 31 positions in the tiled product
        batch.gemm_q8_0_tiled((s(0, 2048), s(1, 128)), s(2, 31 * 128), s(3, 31 * 256), 64, 32, 31, (32, 64))
    with pytest.raises(C.Dispatch):   # 48 rows in the tiled product
        batch.gemm_q8_0_tiled((s(0, 48 * 32), s(1, 96)), s(2, 32 * 128), s(3, 32 * 48 * 4), 48, 32, 32, (32, 48))
    good = ((s(0, 64 * 64), s(1, 64 * 2 * 2)), s(2, 5 * 64 * 4), s(3, 5 * 64 * 4), 64, 64, 5, (64, 64))
    bad = [
        (good[0], good[1], good[2], 0, 64, 5, (64, 64)),                        # no rows
        (good[0], good[1], good[2], 64, 64, 0, (64, 64)),                       # no positions
        (good[0], s(2, 5 * 64 * 4), good[2], 64, 64, 5, (60, 64)),              # x rows closer than cols
        (good[0], s(2, (4 * 66 + 64) * 4), good[2], 64, 64, 5, (66, 64)),       # x stride not a multiple of 4
        (good[0], good[1], good[2], 64, 64, 5, (64, 63)),                       # y rows closer than rows
        ((C.Slice(0, 8, 64 * 64), good[0][1]), good[1], good[2], 64, 64, 5, (64, 64)),   # codes off 16 bytes
        ((good[0][0], s(1, 100)), good[1], good[2], 64, 64, 5, (64, 64)),       # scales of the wrong length
        (good[0], C.Slice(2, 4, 5 * 64 * 4), good[2], 64, 64, 5, (64, 64)),     # x off 16 bytes
        (good[0], good[1], s(0, 5 * 64 * 4), 64, 64, 5, (64, 64)),              # y over the codes
    ]
    for case in bad:
        with pytest.raises(C.Dispatch):
            batch.gemm_q8_0(*case)
    with pytest.raises(C.Dispatch):   # output in resident memory
        att = batch.attach(res)
        batch.gemm_q8_0(good[0], good[1], C.Slice(att.buffer, 0, 5 * 64 * 4), 64, 64, 5, (64, 64))
    with pytest.raises(C.Dispatch):   # bf16 positions: rows of x must stay on 16-byte boundaries (stride % 8)
        batch.gemm_q8_0_bf16(good[0], s(2, (4 * 68 + 64) * 2), good[2], 64, 64, 5, (68, 64))
    with pytest.raises(C.Dispatch):   # bf16 positions: x of the f32 length
        batch.gemm_q8_0_bf16(good[0], good[1], good[2], 64, 64, 5, (64, 64))
    assert batch.dispatches() == 0
    batch.gemm_q8_0(*good)
    assert batch.dispatches() == 1
    batch.gemm_q8_0_bf16(good[0], s(2, 5 * 64 * 2), good[2], 64, 64, 5, (64, 64))
    assert batch.dispatches() == 2
    batch.drop()
    for b in bufs:
        b.free()
    res.free()


def test_split_blocks_host_helper_matches_the_oracle():
    raw = np.random.default_rng(0).integers(0, 256, 34 * 50, dtype=np.uint8)
    codes, scales = C.split_q8_0_blocks(raw.tobytes())
    want_codes, want_scales = orc.q8_split_blocks(raw)
    assert np.array_equal(codes, want_codes) and np.array_equal(scales, want_scales)


@pytest.mark.parametrize("chunk", [1, 40])
def test_tiny_model_golden_with_device_projections(gpu, chunk):
    """Projections (Q8_0), pre-attention step and attention on the device; transformers' logits within 2e-3."""
    model = tm.TinyModel(os.path.join(FIXTURE, "model.gguf"))
    ids, want = tm.load_fixture(FIXTURE)
    held = {}
    for name, (raw, rows, cols) in model.q8_raw.items():
        codes, scales = C.split_q8_0_blocks(raw)
        held[name] = (gpu.resident(codes), gpu.resident(scales), rows, cols)

    def project(name, x):
        codes, scales, rows, cols = held[name]
        n = x.shape[0]
        xb, yb = gpu.upload(x), gpu.buffer(n * rows * 4)
        batch = gpu.batch([xb, yb])
        m = (batch.attach(codes), batch.attach(scales))
        if n == 1:
            batch.gemv_q8_0(m, C.Slice(0, 0, x.nbytes), C.Slice(1, 0, n * rows * 4), rows, cols)
        else:
            batch.gemm_q8_0(m, C.Slice(0, 0, x.nbytes), C.Slice(1, 0, n * rows * 4), rows, cols, n, (cols, rows))
        batch.run()
        batch.drop()
        y = yb.read(np.float32).reshape(n, rows)
        xb.free()
        yb.free()
        return y

    s = DeviceSession(gpu, model, chunk, C.F32, False)
    try:
        got = model.forward(ids, s.prepare, s.attention, chunk=chunk, project=project)
    finally:
        s.close()
        for codes, scales, _, _ in held.values():
            codes.free()
            scales.free()
    assert np.abs(got - want).max() < TOLERANCE


@pytest.mark.parametrize("n", [1, 5, 16, 17, 31, 40])
def test_several_matrices_in_one_dispatch_give_the_separate_products(gpu, n):
    """The q, k and v projections of a layer (gpu.rs:724-732 records three products) as one call: bit for bit
    the three separate gemm_q8_0 products, in one dispatch below 32 positions (three from 32 on); rows that are
    not a multiple of 16, a fourth matrix, and the refusals."""
    cols = 2880
    shapes = [(4096, 21), (512, 22), (37, 23), (528, 24)]
    mats = [q8_test_matrix(rows, cols, seed)[:2] for rows, seed in shapes]
    x = xorshift_values(31 + n, n * cols).reshape(n, cols)
    bufs = [gpu.upload(x)]
    for codes, bits in mats:
        bufs += [gpu.upload(codes), gpu.upload(bits)]
    y_lens = [n * rows * 4 for rows, _ in shapes]
    bufs += [gpu.buffer(2 * sum(y_lens))]                   # all outputs, once per way of computing them
    bufs[-1].fill(0xFF)
    batch = gpu.batch(bufs)
    xs = C.Slice(0, 0, x.nbytes)
    many, offset = [], 0
    for i, ((rows, _), (codes, bits)) in enumerate(zip(shapes, mats)):
        m = (C.Slice(1 + 2 * i, 0, codes.nbytes), C.Slice(2 + 2 * i, 0, bits.nbytes))
        many.append((m, C.Slice(9, offset, y_lens[i]), rows))
        batch.gemm_q8_0(m, xs, C.Slice(9, sum(y_lens) + offset, y_lens[i]), rows, cols, n, (cols, rows))
        offset += y_lens[i]
    before = batch.dispatches()
    batch.gemm_q8_0_many(many, xs, cols, n, cols)
    assert batch.dispatches() - before == (1 if n < 32 else 4)
    # refusals: nothing is recorded
    with pytest.raises(C.Dispatch):
        batch.gemm_q8_0_many(many + many[:1], xs, cols, n, cols)                       # five matrices
    with pytest.raises(C.Dispatch):
        batch.gemm_q8_0_many([], xs, cols, n, cols)
    with pytest.raises(C.Dispatch):
        batch.gemm_q8_0_many([many[0], (many[1][0], many[0][1], many[0][2])], xs, cols, n, cols)   # same output twice
    with pytest.raises(C.Dispatch):
        batch.gemm_q8_0_many([many[0], (many[1][0], many[1][1], 513)], xs, cols, n, cols)          # rows do not fit the slices
    with pytest.raises(C.Dispatch):
        batch.gemm_q8_0_many([(many[0][0], C.Slice(1, 0, y_lens[0]), 4096)], xs, cols, n, cols)     # output over a matrix
    assert batch.dispatches() - before == (1 if n < 32 else 4)
    batch.run()
    raw = bufs[-1].read(np.float32)
    batch.drop()
    for b in bufs:
        b.free()
    together, apart = raw[:raw.size // 2], raw[raw.size // 2:]
    assert not np.isnan(together).any() and np.array_equal(together, apart)


@pytest.mark.parametrize("n,cols", [(1, 2880), (5, 2880), (16, 2880), (31, 2880), (1, 12288), (3, 12288), (2, 32)])
def test_products_of_rms_normalised_positions(gpu, n, cols):
    """gemm_q8_0_many_normed against the reference's sequence (gpu.rs:712-732): copy the hidden rows, normalise the
    copy in place, three products. Within 1e-5 of the largest |y| (the sums of squares are added in another
    order); the hidden rows themselves are not touched; refusals."""
    eps = 1e-5
    shapes = [(4096, 41), (512, 42), (512, 43)] if cols == 2880 else [(80, 41), (64, 42), (37, 43)]
    mats = [q8_test_matrix(rows, cols, seed)[:2] for rows, seed in shapes]
    h = (xorshift_values(51 + n, n * cols) * 3).reshape(n, cols)
    w = 1 + 0.2 * xorshift_values(52, cols)
    bufs = [gpu.upload(h), gpu.buffer(h.nbytes), gpu.upload(w)]
    for codes, bits in mats:
        bufs += [gpu.upload(codes), gpu.upload(bits)]
    y_lens = [n * rows * 4 for rows, _ in shapes]
    bufs += [gpu.buffer(2 * sum(y_lens))]
    batch = gpu.batch(bufs)
    hs, xs, ws = C.Slice(0, 0, h.nbytes), C.Slice(1, 0, h.nbytes), C.Slice(2, 0, w.nbytes)
    batch.copy_rows((hs, cols), (xs, cols), n, cols)
    batch.rmsnorm_rows((xs, ws), n, (cols, cols), eps)
    many, offset = [], 0
    for i, ((rows, _), (codes, bits)) in enumerate(zip(shapes, mats)):
        m = (C.Slice(3 + 2 * i, 0, codes.nbytes), C.Slice(4 + 2 * i, 0, bits.nbytes))
        many.append((m, C.Slice(9, offset, y_lens[i]), rows))
        batch.gemm_q8_0(m, xs, C.Slice(9, sum(y_lens) + offset, y_lens[i]), rows, cols, n, (cols, rows))
        offset += y_lens[i]
    before = batch.dispatches()
    batch.gemm_q8_0_many_normed(many, hs, (ws, eps), cols, n, cols)
    assert batch.dispatches() == before + 1
    with pytest.raises(C.Dispatch):
        batch.gemm_q8_0_many_normed(many, hs, (C.Slice(2, 4, w.nbytes - 4), eps), cols, n, cols)    # weights too short
    with pytest.raises(C.Dispatch):
        batch.gemm_q8_0_many_normed([(many[0][0], C.Slice(2, 0, w.nbytes), 1)], hs, (ws, eps), cols, n, cols)
    assert batch.dispatches() == before + 1
    batch.run()
    raw = bufs[-1].read(np.float32)
    assert np.array_equal(bufs[0].read(np.float32).reshape(n, cols), h)
    batch.drop()
    for b in bufs:
        b.free()
    together, apart = raw[:raw.size // 2], raw[raw.size // 2:]
    assert not np.isnan(together).any()
    assert np.abs(together - apart).max() <= 1e-5 * np.abs(apart).max()


def test_the_normalised_product_is_for_decoding(gpu):
    cols = 64
    codes, bits, _ = q8_test_matrix(64, cols, 3)
    bufs = [gpu.buffer(32 * cols * 4), gpu.upload(np.ones(cols, np.float32)), gpu.upload(codes), gpu.upload(bits),
            gpu.buffer(32 * 64 * 4)]
    batch = gpu.batch(bufs)
    m = [((C.Slice(2, 0, codes.nbytes), C.Slice(3, 0, bits.nbytes)), C.Slice(4, 0, 32 * 64 * 4), 64)]
    with pytest.raises(C.Dispatch, match="fewer than 32"):
        batch.gemm_q8_0_many_normed(m, C.Slice(0, 0, 32 * cols * 4), (C.Slice(1, 0, cols * 4), 1e-5), cols, 32, cols)
    with pytest.raises(C.Dispatch, match="fewer than 32"):
        batch.gemm_q8_0_residual(m[0][0], C.Slice(0, 0, 32 * cols * 4), None, C.Slice(4, 0, 32 * 64 * 4), 64, cols, 32, (cols, 64))
    assert batch.dispatches() == 0
    batch.drop()
    for b in bufs:
        b.free()


@pytest.mark.parametrize("n,bf16", [(1, False), (7, False), (31, False), (1, True), (16, True)])
def test_output_projection_with_bias_and_residual_folded_in(gpu, n, bf16):
    """gemm_q8_0_residual against the reference's three dispatches (gpu.rs:807-827: the product, add_rows of the
    bias, add_rows into the hidden state): the same bits, for f32 and bf16 positions, hidden rows wider than the
    product, with and without a bias."""
    from tests.helpers import to_bf16_bits
    rows, cols, h_stride = 2880, 4096, 2912
    codes, bits, _ = q8_test_matrix(rows, cols, 61)
    x = xorshift_values(62 + n, n * cols).reshape(n, cols)
    xin = to_bf16_bits(x) if bf16 else x
    h = xorshift_values(63, n * h_stride).reshape(n, h_stride)
    bias = xorshift_values(64, rows)
    for with_bias in (True, False):
        bufs = [gpu.upload(codes), gpu.upload(bits), gpu.upload(xin), gpu.upload(h), gpu.upload(h), gpu.upload(bias),
                gpu.buffer(n * rows * 4)]
        batch = gpu.batch(bufs)
        m = (C.Slice(0, 0, codes.nbytes), C.Slice(1, 0, bits.nbytes))
        xs = C.Slice(2, 0, xin.nbytes)
        h_len = ((n - 1) * h_stride + rows) * 4
        if bf16:
            batch.gemm_q8_0_bf16(m, xs, C.Slice(6, 0, n * rows * 4), rows, cols, n, (cols, rows))
        else:
            batch.gemm_q8_0(m, xs, C.Slice(6, 0, n * rows * 4), rows, cols, n, (cols, rows))
        if with_bias:
            batch.add_rows(C.Slice(6, 0, n * rows * 4), (C.Slice(5, 0, rows * 4), 0), n, rows)
        for p in range(n):  # add_rows writes dense rows: one call per row of the wider hidden state
            batch.add_rows(C.Slice(3, p * h_stride * 4, rows * 4), (C.Slice(6, p * rows * 4, rows * 4), rows), 1, rows)
        before = batch.dispatches()
        batch.gemm_q8_0_residual(m, xs, C.Slice(5, 0, rows * 4) if with_bias else None, C.Slice(4, 0, h_len), rows, cols, n,
                                 (cols, h_stride), C.BF16 if bf16 else C.F32)
        assert batch.dispatches() == before + 1
        batch.run()
        apart, together = bufs[3].read(np.float32), bufs[4].read(np.float32)
        batch.drop()
        for b in bufs:
            b.free()
        assert not np.isnan(together).any() and np.array_equal(together, apart)
        assert not np.array_equal(together.reshape(n, h_stride)[:, :rows], h[:, :rows])
        assert np.array_equal(together.reshape(n, h_stride)[:, rows:], h[:, rows:])


@pytest.mark.parametrize("rows,cols,n,bf16", [
    (64, 32, 32, False), (37, 96, 33, False), (300, 160, 64, False), (100, 64, 128, False), (129, 2880, 129, False), (65, 224, 1281, False),
    (64, 16384, 40, False), (64, 16416, 40, False),
    (64, 32, 32, True), (37, 96, 48, True), (300, 160, 49, True), (100, 64, 128, True), (129, 4096, 129, True), (65, 224, 1281, True),
    (64, 16384, 130, True)])
def test_products_whose_wavefronts_share_the_columns(gpu, rows, cols, n, bf16):
    """32 positions or more: the tiles' edges in rows and positions, the positions at which the tile changes, one block,
    an odd number of blocks (a last pair of one), fewer pairs than wavefronts, the widest matrix whose scales LDS holds and
    one wider; scales off a 4-byte boundary; gaps of y untouched. The reference's bound (glue.rs:171), and the kernel of
    256 x 128 tiles within twice the distance of either from float64."""
    from tests.helpers import from_bf16_bits, to_bf16_bits
    codes, bits, elements = q8_test_matrix(rows, cols, 80 + rows)
    x = xorshift_values(23, n * cols).reshape(n, cols)
    xin = to_bf16_bits(x) if bf16 else x
    want = (from_bf16_bits(xin) if bf16 else x).astype(np.float64) @ elements.T
    y_stride = rows + 4
    y_len = ((n - 1) * y_stride + rows) * 4
    bufs = [gpu.upload(codes), gpu.upload(np.concatenate([np.array([0x7E00], np.uint16), bits])), gpu.upload(xin), gpu.buffer(y_len)]
    outs = []
    try:
        for force in ("1", "0"):
            gpu.debug_set("LNG_Q8_MID", force)
            bufs[3].fill(0xFF)
            batch = gpu.batch(bufs)
            m = (C.Slice(0, 0, codes.nbytes), C.Slice(1, 2, bits.nbytes))
            (batch.gemm_q8_0_bf16 if bf16 else batch.gemm_q8_0)(m, C.Slice(2, 0, xin.nbytes), C.Slice(3, 0, y_len), rows, cols, n, (cols, y_stride))
            done = batch.run()
            assert not isinstance(done.gpu_time, Exception), done.gpu_time
            batch.drop()
            out = np.full(n * y_stride, np.nan, np.float32)
            out[:y_len // 4] = bufs[3].read(np.float32)
            outs.append(out.reshape(n, y_stride))
    finally:
        gpu.debug_set("LNG_Q8_MID", None)
    for b in bufs:
        b.free()
    for out in outs:
        assert not np.isnan(out[:, :rows]).any() and np.isnan(out[:-1, rows:]).all()
        assert np.abs(out[:, :rows] - want).max() / np.abs(want).max() < 1e-5
    assert np.abs(outs[0][:, :rows] - outs[1][:, :rows]).max() / np.abs(want).max() < 2e-5


@pytest.mark.parametrize("rows,cols,n,bf16", [
    (1, 32, 1, False), (17, 64, 1, False), (48, 96, 2, False), (33, 224, 15, False), (16, 4128, 16, False), (31, 12288, 1, False),
    (20, 12320, 1, False), (20, 16384, 3, False), (20, 16416, 16, False), (20, 16416, 17, False), (37, 160, 17, False), (300, 2880, 31, False),
    (1, 32, 1, True), (17, 96, 2, True), (33, 224, 16, True), (16, 4128, 1, True), (20, 24576, 1, True), (20, 24608, 1, True),
    (20, 16416, 5, True), (20, 16416, 31, True), (37, 160, 17, True)])
def test_products_of_few_positions(gpu, rows, cols, n, bf16):
    """Fewer than 32 positions: the tiles' edges in rows and positions, one block, an odd number of blocks, fewer pairs of
    blocks than wavefronts, several turns of a wavefront, the widest rows whose x or scales LDS holds and wider ones; scales
    on and off a 4-byte boundary; strided x and y, gaps of y untouched. The reference's bound (glue.rs:171)."""
    from tests.helpers import from_bf16_bits, to_bf16_bits
    codes, bits, elements = q8_test_matrix(rows, cols, 90 + rows)
    x = np.full((n, cols + 8), np.nan, np.float32)
    x[:, :cols] = xorshift_values(29, n * cols).reshape(n, cols)
    xin = to_bf16_bits(x) if bf16 else x
    want = (from_bf16_bits(xin) if bf16 else x)[:, :cols].astype(np.float64) @ elements.T
    y_stride = rows + 4
    y_len = ((n - 1) * y_stride + rows) * 4
    for shift in (0, 2):
        bufs = [gpu.upload(codes), gpu.upload(np.concatenate([np.full(shift // 2, 0x7E00, np.uint16), bits])), gpu.upload(xin), gpu.buffer(y_len)]
        bufs[3].fill(0xFF)
        batch = gpu.batch(bufs)
        m = (C.Slice(0, 0, codes.nbytes), C.Slice(1, shift, bits.nbytes))
        xs = C.Slice(2, 0, ((n - 1) * (cols + 8) + cols) * (2 if bf16 else 4))
        (batch.gemm_q8_0_bf16 if bf16 else batch.gemm_q8_0)(m, xs, C.Slice(3, 0, y_len), rows, cols, n, (cols + 8, y_stride))
        done = batch.run()
        assert not isinstance(done.gpu_time, Exception), done.gpu_time
        out = np.full(n * y_stride, np.nan, np.float32)
        out[:y_len // 4] = bufs[3].read(np.float32)
        batch.drop()
        for b in bufs:
            b.free()
        out = out.reshape(n, y_stride)
        assert not np.isnan(out[:, :rows]).any() and np.isnan(out[:-1, rows:]).all()
        assert np.abs(out[:, :rows] - want).max() / np.abs(want).max() < 1e-5


@pytest.mark.parametrize("n", [33, 128, 200, 700])
def test_matrices_of_many_rows_among_others(gpu, n):
    """32 positions or more: a matrix whose tiles of 256 x 128 fill the device and two that leave it mostly idle, in one call
    and each alone: the same bits, within the reference's bound (glue.rs:171) of float64."""
    cols = 64
    shapes = [(96, 7), (20000, 8), (513, 9)]
    x = xorshift_values(41, n * cols).reshape(n, cols)
    mats = [q8_test_matrix(rows, cols, seed) for rows, seed in shapes]
    y_lens = [n * rows * 4 for rows, _ in shapes]
    bufs = [gpu.upload(x)]
    for codes, bits, _ in mats:
        bufs += [gpu.upload(codes), gpu.upload(bits)]
    bufs += [gpu.buffer(2 * sum(y_lens))]
    bufs[-1].fill(0xFF)
    batch = gpu.batch(bufs)
    xs, many, offset = C.Slice(0, 0, x.nbytes), [], 0
    for i, ((rows, _), (codes, bits, _)) in enumerate(zip(shapes, mats)):
        m = (C.Slice(1 + 2 * i, 0, codes.nbytes), C.Slice(2 + 2 * i, 0, bits.nbytes))
        many.append((m, C.Slice(7, offset, y_lens[i]), rows))
        batch.gemm_q8_0(m, xs, C.Slice(7, sum(y_lens) + offset, y_lens[i]), rows, cols, n, (cols, rows))
        offset += y_lens[i]
    batch.gemm_q8_0_many(many, xs, cols, n, cols)
    done = batch.run()
    assert not isinstance(done.gpu_time, Exception), done.gpu_time
    raw = bufs[-1].read(np.float32)
    batch.drop()
    for b in bufs:
        b.free()
    together, alone = raw[:raw.size // 2], raw[raw.size // 2:]
    assert not np.isnan(together).any() and np.array_equal(together, alone)
    offset = 0
    for (rows, _), (_, _, elements) in zip(shapes, mats):
        want = x.astype(np.float64) @ elements.T
        assert np.abs(alone[offset:offset + n * rows].reshape(n, rows) - want).max() / np.abs(want).max() < 1e-5
        offset += n * rows


def _product(gpu, codes, bits, xin, rows, cols, n, norm=None):
    """y[n][rows] of the first `rows` rows of a matrix."""
    bufs = [gpu.upload(codes), gpu.upload(bits), gpu.upload(xin), gpu.buffer(n * rows * 4)] + ([gpu.upload(norm)] if norm is not None else [])
    bufs[3].fill(0xFF)
    batch = gpu.batch(bufs)
    m, xs, ys = (C.Slice(0, 0, rows * cols), C.Slice(1, 0, rows * cols // 16)), C.Slice(2, 0, xin.nbytes), C.Slice(3, 0, n * rows * 4)
    if norm is not None:
        batch.gemm_q8_0_many_normed([(m, ys, rows)], xs, (C.Slice(4, 0, cols * 4), 1e-5), cols, n, cols)
    else:
        (batch.gemm_q8_0_bf16 if xin.dtype == np.uint16 else batch.gemm_q8_0)(m, xs, ys, rows, cols, n, (cols, rows))
    done = batch.run()
    assert not isinstance(done.gpu_time, Exception), done.gpu_time
    y = bufs[3].read(np.float32).reshape(n, rows)
    batch.drop()
    for b in bufs:
        b.free()
    return y


@pytest.mark.parametrize("cols,n,bf16", [(32, 2, False), (96, 16, False), (224, 17, False), (512, 31, False), (1152, 16, False),
                                         (96, 17, True), (512, 31, True)])
def test_few_positions_give_the_same_bits_in_every_kernel(gpu, cols, n, bf16):
    """A few rows and all rows of one matrix: split by the product itself and before it, in tiles of 16 rows and of 32 x 32
    (16 x 32 from bf16), with whole pairs of blocks and a block left over; within the reference's bound (glue.rs:171) of float64."""
    from tests.helpers import from_bf16_bits, to_bf16_bits
    rows, few = 9000, 40
    codes, bits, elements = q8_test_matrix(rows, cols, 30 + cols)
    x = xorshift_values(43, n * cols).reshape(n, cols)
    xin = to_bf16_bits(x) if bf16 else x
    want = (from_bf16_bits(xin) if bf16 else x).astype(np.float64) @ elements.T
    whole, part = _product(gpu, codes, bits, xin, rows, cols, n), _product(gpu, codes, bits, xin, few, cols, n)
    assert np.array_equal(whole[:, :few], part)
    assert np.abs(whole - want).max() / np.abs(want).max() < 1e-5


@pytest.mark.parametrize("rows,cols,n", [(40, 32, 2), (100, 512, 8), (37, 512, 9), (16, 512, 16), (2100, 96, 17), (300, 256, 31), (33, 2048, 4), (5000, 512, 8)])
def test_positions_normalised_by_the_product_itself(gpu, rows, cols, n):
    """Narrow matrices of up to 31 positions: one wavefront and both take a position's sum of squares, groups of 16 positions;
    within the reference's bound (glue.rs:171) of float64."""
    codes, bits, elements = q8_test_matrix(rows, cols, 50 + cols)
    x, w = 3 * xorshift_values(44, n * cols).reshape(n, cols), 1 + 0.2 * xorshift_values(45, cols)
    xd = x.astype(np.float64)
    want = (xd / np.sqrt((xd * xd).mean(axis=1, keepdims=True) + 1e-5) * w) @ elements.T
    got = _product(gpu, codes, bits, x, rows, cols, n, w)
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-5


@pytest.mark.parametrize("rows,cols,bf16", [(1, 32, False), (37, 96, False), (130, 4128, False), (2880, 4096, False), (5120, 2880, False), (8200, 64, False),
                                            (33, 12288, False), (9, 32, True), (2880, 4096, True), (3600, 160, True), (40, 24576, True)])
def test_one_position_in_whole_numbers(gpu, rows, cols, bf16):
    """lng_q8_one takes a block of x as 30-bit whole numbers of a unit of its own: tiles of 8 to 16 rows and their remainders,
    one block, an odd number of blocks, several turns, values of a block far apart, blocks from the smallest normal numbers to
    2^60. Every sum is exact within a block; per output at most 6 roundings of a block's value, blocks / 32 + 1 of a lane's sum and
    10 of the lanes' and wavefronts', each 2^-24 of the terms, and 2^-30 of a block's largest x for each x. NaN makes the outputs
    NaN, an infinity too from f32 (the lower of its two bf16 values is NaN); from bf16 it gives infinities, and NaN where the code
    is 0, as two positions of it do."""
    from tests.helpers import from_bf16_bits, to_bf16_bits
    codes, bits, elements = q8_test_matrix(rows, cols, 90 + rows)
    blocks = cols // 32
    rng = np.random.default_rng(rows + cols)
    for spread, units in ((0, np.zeros(blocks)), (24, rng.integers(-126, 60, blocks))):
        x = xorshift_values(31, cols).reshape(blocks, 32) * np.exp2(-rng.integers(0, spread + 1, (blocks, 32))) * np.exp2(units)[:, None]
        xin = to_bf16_bits(x.astype(np.float32).reshape(1, cols)) if bf16 else x.astype(np.float32).reshape(1, cols)
        exact = (from_bf16_bits(xin) if bf16 else xin).astype(np.float64)
        outs = [_product(gpu, codes, bits, xin, rows, cols, 1)]
        want = exact @ elements.T
        terms = np.abs(exact) @ np.abs(elements).T
        largest = np.abs(exact).reshape(blocks, 32).max(1) @ np.abs(elements).reshape(rows, blocks, 32).sum(2).T
        bound = (17 + blocks / 32) * 2.0**-24 * terms[0] + 2.0**-30 * largest + (blocks + 32) * 2.0**-140  # (the last: f32's own end)
        assert (np.abs(outs[0][0] - want[0]) <= bound).all()
    for bad in (np.inf, np.nan):
        x = xorshift_values(32, cols).astype(np.float32).reshape(1, cols)
        x[0, cols - 5] = bad
        got = _product(gpu, codes, bits, to_bf16_bits(x) if bf16 else x, rows, cols, 1)
        if not bf16 or np.isnan(bad):
            assert np.isnan(got).all()
        else:
            column = elements[:, cols - 5]  # (code times scale, which may be negative)
            assert np.array_equal(got[0], np.where(column == 0, np.nan, np.copysign(np.inf, column)), equal_nan=True)
            assert np.array_equal(got.repeat(2, 0), _product(gpu, codes, bits, to_bf16_bits(x.repeat(2, 0)), rows, cols, 2), equal_nan=True)


@pytest.mark.parametrize("rows,cols,bf16", [(40, 32, False), (2880, 4096, False), (5120, 2880, False), (130, 4128, False), (70, 160, False), (33, 8192, False), (33, 8224, False), (33, 12288, False),
                                            (40, 32, True), (2880, 4096, True), (130, 5152, True), (40, 24576, True)])
@pytest.mark.parametrize("outlier", [2.0**13, 2.0**20, 2.0**31, 2.0**45, 2.0**90])
def test_one_position_of_values_far_apart(gpu, rows, cols, bf16, outlier):
    """One x of each block is `outlier` times the others, and every other row has the code 0 there, so that all of its result is of the
    small ones. An x counts with 2^-18 of itself (two bf16 values; bf16 positions: exactly) whatever else its block holds, a bf16
    value below 2^-126 perhaps as zero; the sums round at most 64 times within a block and blocks / 32 + 16 times after it. With a
    norm too, whose own roundings are eight of each x."""
    from tests.helpers import from_bf16_bits, to_bf16_bits
    codes, bits, elements = q8_test_matrix(rows, cols, 60 + rows)
    blocks = cols // 32
    rng = np.random.default_rng(rows + cols)
    at = np.arange(blocks) * 32 + rng.integers(0, 32, blocks)
    codes = codes.reshape(rows, cols).copy()
    elements = elements.copy()
    codes[::2, at] = 0
    elements[::2, at] = 0.0
    x = xorshift_values(36, cols).astype(np.float32) * 2.0**-20
    x[at] *= np.float32(outlier)
    w = np.exp2(np.floor(rng.random(cols) * 3)).astype(np.float32)
    xin = (to_bf16_bits(x) if bf16 else x).reshape(1, cols)
    exact = (from_bf16_bits(xin) if bf16 else xin)[0].astype(np.float64)
    for norm in (None,) if bf16 or outlier > 2.0**60 else (None, w):
        xs = exact if norm is None else exact / np.sqrt((exact * exact).mean() + 1e-5) * norm
        got = _product(gpu, codes.reshape(-1), bits, xin, rows, cols, 1, norm)[0]
        terms = np.abs(elements) @ np.abs(xs)
        bound = ((0 if bf16 else 2.0**-18) + (80 + blocks / 32 + (0 if norm is None else 8)) * 2.0**-24) * terms + np.abs(elements).sum(1) * 2.0**-126
        assert (np.abs(got - elements @ xs) <= bound).all(), np.max(np.abs(got - elements @ xs) / bound)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("rows,cols", [(40, 1024), (40, 1056), (37, 1536), (300, 1568), (5120, 2048), (33, 2080), (2880, 2560), (33, 2592), (17, 6176)])
def test_one_position_at_the_edges_of_what_is_in_flight(gpu, rows, cols, bf16):
    """Columns either side of the numbers of pairs of blocks that a wavefront asks for at once, odd numbers of pairs and of blocks
    among them; the bound of test_one_position_in_whole_numbers."""
    from tests.helpers import from_bf16_bits, to_bf16_bits
    codes, bits, elements = q8_test_matrix(rows, cols, 70 + rows)
    x = xorshift_values(37, cols).astype(np.float32).reshape(1, cols)
    xin = to_bf16_bits(x) if bf16 else x
    exact = (from_bf16_bits(xin) if bf16 else xin)[0].astype(np.float64)
    got = _product(gpu, codes, bits, xin, rows, cols, 1)[0]
    largest = np.abs(elements).reshape(rows, cols // 32, 32).sum(2) @ np.abs(exact).reshape(cols // 32, 32).max(1)
    assert (np.abs(got - elements @ exact) <= (17 + cols / 1024) * 2.0**-24 * (np.abs(elements) @ np.abs(exact)) + 2.0**-30 * largest).all()


@pytest.mark.parametrize("kind", ["f32", "norm", "bf16"])
@pytest.mark.parametrize("rows,cols", [(8193, 32), (9001, 96), (12290, 1024), (16400, 1056), (8195, 2080), (8200, 3104), (8210, 4128), (4100, 12288)])
def test_one_position_of_many_rows(gpu, rows, cols, kind):
    """More tiles than the device holds workgroups: each workgroup takes several, the last of them fewer rows; every number of pairs in
    flight, one workgroup a unit too (12,288 columns). Bit for bit what parts of the matrix give that are a workgroup to a tile - an
    output's sum knows nothing of the other rows - with values far apart in every block; and within the reference's bound (glue.rs:171)
    of float64."""
    from tests.helpers import from_bf16_bits, to_bf16_bits
    codes, bits, elements = q8_test_matrix(rows, cols, 91)
    x = xorshift_values(38, cols).astype(np.float32)
    x[5::32] *= np.float32(2.0**28)
    x[9::64] *= np.float32(2.0**-14)
    xin = (to_bf16_bits(x) if kind == "bf16" else x).reshape(1, cols)
    w = xorshift_values(39, cols).astype(np.float32) + 1.0 if kind == "norm" else None
    got = _product(gpu, codes, bits, xin, rows, cols, 1, w)[0]
    step = 2000
    for at in range(0, rows, step):
        part = min(step, rows - at)
        assert np.array_equal(got[at:at + part], _product(gpu, codes[at * cols:][:part * cols], bits[at * cols // 32:][:part * cols // 32], xin, part, cols, 1, w)[0])
    exact = (from_bf16_bits(xin) if kind == "bf16" else xin)[0].astype(np.float64)
    if kind == "norm":
        exact = exact / np.sqrt((exact * exact).mean() + 1e-5) * w
    want = elements @ exact
    assert np.abs(got - want).max() / np.abs(want).max() < 1e-5


def test_one_position_of_many_rows_in_several_matrices_and_added(gpu):
    """Several matrices whose tiles together are more than the device holds workgroups, and one such with bias and residual: bit for bit
    each matrix alone, and the sums of the separate dispatches."""
    cols, shapes = 288, [5003, 64, 4200]
    mats = [q8_test_matrix(r, cols, 92 + i) for i, r in enumerate(shapes)]
    x = xorshift_values(46, cols).astype(np.float32).reshape(1, cols)
    bufs = [gpu.upload(x)] + [gpu.upload(a) for m in mats for a in m[:2]] + [gpu.buffer(4 * sum(shapes))]
    bufs[-1].fill(0xFF)
    batch = gpu.batch(bufs)
    starts = [0] + list(np.cumsum(shapes))
    batch.gemm_q8_0_many([((C.Slice(1 + 2 * i, 0, r * cols), C.Slice(2 + 2 * i, 0, r * cols // 16)), C.Slice(7, 4 * int(starts[i]), 4 * r), r)
                          for i, r in enumerate(shapes)], C.Slice(0, 0, cols * 4), cols, 1, cols)
    done = batch.run()
    assert not isinstance(done.gpu_time, Exception), done.gpu_time
    got = bufs[-1].read(np.float32)
    batch.drop()
    for b in bufs:
        b.free()
    for i, r in enumerate(shapes):
        assert np.array_equal(got[starts[i]:starts[i + 1]], _product(gpu, mats[i][0], mats[i][1], x, r, cols, 1)[0])
    rows = 9001
    codes, bits, _ = q8_test_matrix(rows, cols, 96)
    bias, h = xorshift_values(47, rows).astype(np.float32), xorshift_values(48, rows).astype(np.float32)
    y = _product(gpu, codes, bits, x, rows, cols, 1)[0]
    bufs = [gpu.upload(a) for a in (codes, bits, x, bias, h)]
    batch = gpu.batch(bufs)
    batch.gemm_q8_0_residual((C.Slice(0, 0, rows * cols), C.Slice(1, 0, rows * cols // 16)), C.Slice(2, 0, cols * 4), C.Slice(3, 0, rows * 4), C.Slice(4, 0, rows * 4), rows, cols, 1, (cols, rows))
    done = batch.run()
    assert not isinstance(done.gpu_time, Exception), done.gpu_time
    assert np.array_equal(bufs[4].read(np.float32), h + (y + bias))
    batch.drop()
    for b in bufs:
        b.free()


@pytest.mark.parametrize("rows,cols,n", [(4098, 2048, 2), (4100, 2080, 16), (5120, 2880, 9), (5121, 3104, 3), (8192, 4096, 16), (8150, 4064, 15), (7000, 2048, 3)])
def test_positions_split_by_the_product_itself(gpu, rows, cols, n):
    """2 to 16 f32 positions of more rows than compute units have 16 for, one dispatch with and without the RMS norm: workgroups of 18
    to 32 rows and their remainders, an odd number of blocks, wavefronts with a pair fewer than others, one column size either side
    of the two numbers of pairs a wavefront holds; positions of very different sizes; scales off a 4-byte boundary. Within the
    reference's bound (glue.rs:171) of float64 at each position."""
    codes, bits, elements = q8_test_matrix(rows, cols, 33 + rows)
    x = (xorshift_values(34 + n, n * cols).reshape(n, cols) * (10.0 ** np.arange(-8, 8))[:n, None]).astype(np.float32)
    w = xorshift_values(35, cols).astype(np.float32) + 1.0
    normed = x.astype(np.float64) / np.sqrt((x.astype(np.float64) ** 2).mean(1, keepdims=True) + 1e-5) * w
    bufs = [gpu.upload(codes), gpu.upload(np.concatenate([np.array([0x7E00], np.uint16), bits])), gpu.upload(x), gpu.upload(w), gpu.buffer(n * rows * 4), gpu.buffer(n * rows * 4)]
    for b in bufs[4:]:
        b.fill(0xFF)
    batch = gpu.batch(bufs)
    batch.set_timing(True)
    m, xs = (C.Slice(0, 0, codes.nbytes), C.Slice(1, 2, bits.nbytes)), C.Slice(2, 0, x.nbytes)
    batch.gemm_q8_0(m, xs, C.Slice(4, 0, n * rows * 4), rows, cols, n, (cols, rows))
    batch.gemm_q8_0_many_normed([(m, C.Slice(5, 0, n * rows * 4), rows)], xs, (C.Slice(3, 0, w.nbytes), 1e-5), cols, n, cols)
    done = batch.run()
    assert not isinstance(done.gpu_time, Exception), done.gpu_time
    assert batch.kernel_seconds("lng_q8_few_split")[1] == 2 and batch.dispatches() == 2
    batch.drop()
    for buf, values in ((bufs[4], x.astype(np.float64)), (bufs[5], normed)):
        want, got = values @ elements.T, buf.read(np.float32).reshape(n, rows)
        assert (np.abs(got - want).max(1) < 1e-5 * np.abs(want).max(1)).all()
    for b in bufs:
        b.free()


@pytest.mark.parametrize("normed", [False, True])
@pytest.mark.parametrize("n,cols", [(1, 2880), (2, 2880), (9, 2080), (16, 2880), (16, 4096)])
def test_a_few_positions_together_and_alone(gpu, n, cols, normed):
    """q, k and v in one dispatch, whose rows together decide on the kernel, and each alone. Without a norm bit for bit. With one the
    kernel for many rows multiplies what the norm's weights give and scales the finished sum: both within 2^-17 of float64 for each
    term - two bf16 values hold 2^-18 of each, which leaves as much for the f32 sums of 128 blocks - so neither is the less exact."""
    shapes = [4096, 512, 520]
    mats = [q8_test_matrix(rows, cols, 21 + i) for i, rows in enumerate(shapes)]
    x, w = xorshift_values(49, n * cols).reshape(n, cols).astype(np.float32), 1 + 0.2 * xorshift_values(50, cols).astype(np.float32)
    eps, starts = 1e-5, [0] + list(np.cumsum(shapes) * n * 4)
    bufs = [gpu.upload(x), gpu.upload(w)] + [gpu.upload(a) for m in mats for a in m[:2]] + [gpu.buffer(int(starts[-1]))]
    bufs[-1].fill(0xFF)
    batch = gpu.batch(bufs)
    many = [((C.Slice(2 + 2 * i, 0, r * cols), C.Slice(3 + 2 * i, 0, r * cols // 16)), C.Slice(8, int(starts[i]), 4 * n * r), r) for i, r in enumerate(shapes)]
    xs = C.Slice(0, 0, x.nbytes)
    batch.gemm_q8_0_many_normed(many, xs, (C.Slice(1, 0, w.nbytes), eps), cols, n, cols) if normed else batch.gemm_q8_0_many(many, xs, cols, n, cols)
    done = batch.run()
    assert not isinstance(done.gpu_time, Exception), done.gpu_time
    raw = bufs[-1].read(np.float32)
    batch.drop()
    for b in bufs:
        b.free()
    xd = x.astype(np.float64)
    if normed:
        xd = xd / np.sqrt((xd * xd).mean(axis=1, keepdims=True) + eps) * w
    for i, rows in enumerate(shapes):
        together = raw[starts[i] // 4:starts[i + 1] // 4].reshape(n, rows)
        alone = _product(gpu, mats[i][0], mats[i][1], x, rows, cols, n, w if normed else None)
        if not normed:
            assert np.array_equal(together, alone)
        want, terms = xd @ mats[i][2].T, np.abs(xd) @ np.abs(mats[i][2]).T
        for got in (together, alone):
            assert (np.abs(got - want) <= 2.0**-17 * terms).all(), np.max(np.abs(got - want) / terms) * 2.0**17
