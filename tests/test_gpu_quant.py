"""GPU parity of the quant::* path against the CPU oracle, through the C ABI.

Bar: quantised i8 values, f32 scales, i32 accumulators and the f32 outputs of the W8A8
product are all BIT-EXACT (the epilogue keeps the reference's multiplication order, so
even the f32 result has a single correct bit pattern).
"""
import ctypes as C
import sys

import numpy as np
import pytest

import helpers as H
from devbuf import DevBuf

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def edge_rows(cols):
    """Rows the reference's arithmetic treats specially (ties, zero, NaN, inf, subnormal)."""
    r = np.zeros((6, cols), np.float32)
    r[0, :8] = [127, -127, 0.5, -0.5, 1.5, 2.5, -2.5, 0]
    r[2, :] = 4.0
    r[2, 1::2] = -4.0
    r[3, :8] = [np.nan, 1, -2, 0.5, 0, 0, 0, 2]
    r[4, :8] = [np.inf, 1, -1, 0, 0, 0, 0, -np.inf]
    r[5, :8] = [1e-42, -1e-42, 0, 0, 0, 0, 0, 5e-43]
    return r


@pytest.mark.parametrize("rows,cols", [(32, 4096), (1, 4096), (1, 14336), (7, 100), (5, 4100),
                                       (3, 20000), (2, 16384), (9, 33), (4, 1)])
def test_quantize_activations_bit_exact(ctx, orc, rows, cols):
    from peregrine_amd import quant
    say(f"quantize_activations rows={rows} cols={cols}")
    a = orc.rng_normal(1000 + rows * 7 + cols, rows * cols).reshape(rows, cols)
    a[:, :: max(1, cols // 40)] *= 20  # outlier channels
    q, s = quant.quantize_activations(a, rows, cols, ctx)
    qo, so = orc.quantize_activations(a, rows, cols)
    assert (bits(s) == bits(so)).all()
    assert (q == qo).all()


def test_quantize_activations_edge_rows_and_empty(ctx, orc):
    from peregrine_amd import quant
    for cols in (8, 64, 4096):
        say(f"quantize_activations edge rows cols={cols}")
        a = edge_rows(cols)
        q, s = quant.quantize_activations(a, a.shape[0], cols, ctx)
        qo, so = orc.quantize_activations(a, a.shape[0], cols)
        assert (bits(s) == bits(so)).all() and (q == qo).all()
    # constructed near-tie rows that separate x*(1/s) from x/s
    fh = float.fromhex
    tie = np.array([[fh("0x1.13c502p-4"), fh("0x1.e6658ep-10"), fh("-0x1.09ff8ap-4"), fh("-0x1.f9f07ep-5")],
                    [fh("0x1.18d40ep-5"), fh("0x1.1b0a2p-13"), fh("-0x1.1116c6p-5"), fh("-0x1.134cdap-5")]], np.float32)
    q, s = quant.quantize_activations(tie, 2, 4, ctx)
    qo, so = orc.quantize_activations(tie, 2, 4)
    assert (q == qo).all() and (bits(s) == bits(so)).all()
    q, s = quant.quantize_activations(np.zeros(0, np.float32), 0, 16, ctx)  # empty input
    assert q.size == 0 and s.size == 0
    with pytest.raises(ValueError):
        quant.quantize_activations(np.zeros(5, np.float32), 2, 3, ctx)


@pytest.mark.parametrize("cols", [64, 1028, 1531, 5000])  # less than a wavefront's vectors, a tail of its own, and a workgroup of 1024
def test_quantize_activations_around_every_half(ctx, orc, cols):
    """Half away from zero, at a scale of one: every k + 0.5 of either sign with the floats next to it, where the rounding has its edges."""
    from peregrine_amd import quant
    half = np.arange(-127, 127, dtype=np.float32) + np.float32(0.5)
    v = np.concatenate([np.nextafter(half, np.float32(-np.inf)), half, np.nextafter(half, np.float32(np.inf))]).astype(np.float32)
    a = np.resize(v, (-(-v.size // (cols - 1)), cols - 1))
    a = np.concatenate([np.full((a.shape[0], 1), 127.0, np.float32), a], 1)
    qg, sg = quant.quantize_activations(a, a.shape[0], cols, ctx)
    qc, sc = orc.quantize_activations(a, a.shape[0], cols)
    assert (np.asarray(sg) == 1.0).all() and (np.asarray(sc) == 1.0).all()
    assert (np.asarray(qg).reshape(-1) == np.asarray(qc).reshape(-1)).all()


@pytest.mark.parametrize("rows,cols", [(128, 96), (100, 70), (4096, 64), (64, 1000), (1, 5), (300, 1)])
def test_quantize_weights_bit_exact(ctx, orc, rows, cols):
    from peregrine_amd import quant
    say(f"quantize_weights rows={rows} cols={cols}")
    w = orc.rng_normal(5678 + rows + cols, rows * cols, 0.0, 0.02)
    qt = quant.quantize_weights(w, rows, cols, ctx)
    q, q_t, s = orc.quantize_weights(w, rows, cols)
    assert (bits(qt.scales) == bits(s)).all()
    assert (qt.data_i8 == q).all()
    assert (qt.data_i8_t == q_t).all()
    assert (bits(quant.dequantize(qt, ctx)) == bits(orc.dequantize(q, s, rows, cols))).all()


def test_quantize_weights_edge_columns(ctx, orc):
    from peregrine_amd import quant
    say("quantize_weights edge columns")
    fh = float.fromhex
    w = np.zeros((6, 7), np.float32)
    w[:, 0] = [127, -127, 2.5, -2.5, 0.5, 1.5]
    w[:, 2] = [3, 3, -3, 3, -3, 3]
    w[:, 3] = [np.nan, 1, -2, 0.25, 0, 2]
    w[:, 4] = [np.inf, 1, -1, 0, 5, -np.inf]
    w[:4, 5] = [fh("0x1.13c502p-4"), fh("0x1.e6658ep-10"), fh("-0x1.09ff8ap-4"), fh("-0x1.f9f07ep-5")]
    w[:4, 6] = [fh("0x1.18d40ep-5"), fh("0x1.1b0a2p-13"), fh("-0x1.1116c6p-5"), fh("-0x1.134cdap-5")]
    qt = quant.quantize_weights(w, 6, 7, ctx)
    q, q_t, s = orc.quantize_weights(w, 6, 7)
    assert (bits(qt.scales) == bits(s)).all() and (qt.data_i8 == q).all() and (qt.data_i8_t == q_t).all()


def test_reference_roundtrip_property(ctx):
    # tests/quant_parity.rs:6-32 run against the GPU path
    from peregrine_amd import quant
    rows, cols = 64, 128
    data = H.mod_pattern(rows * cols, 17, 5, 400, 100.0, 2.0)
    qt = quant.quantize_weights(data, rows, cols, ctx)
    rec = quant.dequantize(qt, ctx).reshape(rows, cols)
    d = data.reshape(rows, cols)
    amax = np.abs(d).max(axis=0)
    scale = np.where(amax == 0, 1.0, amax / np.float32(127)).astype(np.float32)
    assert (np.abs(d - rec) <= scale[None, :] + 1e-7).all()


def test_to_gpu_from_gpu_roundtrip(ctx, orc):
    # QuantizedTensor::to_gpu / from_gpu (src/quant.rs:173-191); upload is idempotent
    from peregrine_amd import quant
    rows, cols = 200, 130
    w = orc.rng_normal(77, rows * cols, 0.0, 0.02)
    qt = quant.quantize_weights(w, rows, cols, ctx)
    q0, qt0, s0 = qt.data_i8.copy(), qt.data_i8_t.copy(), qt.scales.copy()
    qt.to_gpu(ctx)
    h = qt._gpu
    qt.to_gpu(ctx)
    assert qt._gpu is h
    qt.data_i8[:] = 0
    qt.from_gpu(ctx)
    assert (qt.data_i8 == q0).all() and (qt.data_i8_t == qt0).all() and (bits(qt.scales) == bits(s0)).all()
    with pytest.raises(RuntimeError):
        quant.matmul_quantized_gpu(ctx, np.zeros(rows, np.float32), 1, rows,
                                   quant.QuantizedTensor(q0, qt0, s0, rows, cols))  # "weights not on GPU"


def run_matmul_dev(ctx, a, m, k, qt):
    """pg_matmul_quantized_dev with the accumulator dump; returns (out, acc)."""
    from peregrine_amd import _ffi
    qt.to_gpu(ctx)
    n = qt.cols
    da = DevBuf(ctx, host=np.ascontiguousarray(a, np.float32))
    dout, dacc = DevBuf(ctx, m * n * 4), DevBuf(ctx, m * n * 4)
    _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr, dacc.ptr))
    ctx.sync()
    return dout.to_host(np.float32), dacc.to_host(np.int32)


# (m, k, n): reference test shapes, decode GEMV shapes, every GEMM tile config, ragged edges
MATMUL_SHAPES = [
    (32, 128, 64), (16, 64, 32),                       # tests/quant_parity.rs:35, src/quant.rs:252
    (8, 32, 16), (1, 64, 1), (16, 256, 32),            # tests/huffman_parity.rs:25
    (1, 4096, 14336), (1, 14336, 4096),                # benchmark configuration 2 (decode GEMV)
    (2, 4096, 1024), (3, 1000, 77), (4, 4096, 300),    # GEMV with m = 2..4, ragged k and n
    (32, 4096, 4096),                                  # benchmark configuration 1
    (5, 96, 40), (64, 200, 130), (65, 384, 129),       # 64x64 and 128x128 tiles, ragged
    (196, 768, 3072), (196, 1024, 4096),               # benches/wallclock.rs:758-786
    (300, 512, 1000),                                  # 128x128 tiles, ragged m and n
    (2048, 128, 4096),                                 # 128x256 tiles
    (2050, 192, 4100),                                 # 128x256 tiles, ragged m and n
    (2049, 128, 12300),                                # 256x256 tiles, ragged m and n
    (1030, 256, 4000),                                 # 128x128 tiles unsplit, ragged m and n
    # 2 .. 32 rows: one launch, a workgroup per 16 (or 32) weight rows with its wavefronts on runs of K (ragged everywhere;
    # K of one unit of 128; more than 16 rows on a wide tensor: two weight tiles per workgroup)
    (5, 4096, 1000), (17, 4224, 520), (31, 512, 77), (2, 128, 16), (16, 130, 5), (9, 2000, 33), (20, 1024, 8200),
    (32, 4096, 14336), (17, 384, 8208), (24, 14336, 4096), (3, 14336, 4100),
    # 33 .. 64 rows on products at least as wide as long: the same with four activation tiles a unit
    (33, 1024, 4100), (40, 1024, 14336), (64, 4096, 4096), (50, 384, 8300),
    # 33 .. 64 rows on long, narrow products: K split over workgroups, i32 partial planes, finishing pass
    (64, 14336, 300), (40, 8192, 4096),
    (100, 8192, 300), (130, 4096, 257), (256, 2048, 1000),   # up to 256 rows when K >= 2 N: 128-row tiles
]


@pytest.mark.parametrize("m,k,n", MATMUL_SHAPES)
def test_matmul_quantized_bit_exact(ctx, orc, m, k, n):
    from peregrine_amd import quant
    say(f"matmul_quantized m={m} k={k} n={n}")
    a = orc.rng_normal(1234 + m, m * k)
    if k >= 100:
        a.reshape(m, k)[:, :: k // 50] *= 20  # outlier channels
    w = orc.rng_normal(5678 + n, k * n, 0.0, 0.02)
    qt = quant.quantize_weights(w, k, n, ctx)
    q, q_t, s = orc.quantize_weights(w, k, n)
    assert (qt.data_i8_t == q_t).all()
    want, want_acc = orc.matmul_quantized(a, m, k, q_t, s, n)
    got, got_acc = run_matmul_dev(ctx, a, m, k, qt)
    assert (got_acc == want_acc).all(), "i32 accumulators differ"
    assert (bits(got) == bits(want)).all(), "f32 outputs differ"
    # the host-pointer entry point gives the same answer
    got2 = quant.matmul_quantized(a, m, k, qt, ctx)
    assert (bits(got2) == bits(want)).all()


@pytest.mark.parametrize("k,n", [(8, 5), (64, 33), (4096, 300), (4100, 64), (14336, 128), (16384, 16), (16400, 16)])
def test_matmul_quantized_one_row_quantised_inside_the_product(ctx, orc, k, n):
    """m = 1 with k % 4 == 0 and k <= 16384 runs as ONE launch that quantises the activation row
    itself: the accumulators (hence the row's integers) and the f32 output must be those of the
    two-step path bit for bit, on ordinary rows and on the rows the arithmetic treats specially
    (ties, zero row, NaN, inf, subnormals).  k = 4100 and 16400 are past that route's limits."""
    from peregrine_amd import quant
    say(f"matmul_quantized one row k={k} n={n}")
    w = orc.rng_normal(321 + n, k * n, 0.0, 0.02)
    qt = quant.quantize_weights(w, k, n, ctx)
    q, q_t, s = orc.quantize_weights(w, k, n)
    rows = [orc.rng_normal(77 + k, k)]
    rows[0][:: max(1, k // 40)] *= 20
    rows += list(edge_rows(k))
    for i, a in enumerate(rows):
        want, want_acc = orc.matmul_quantized(a, 1, k, q_t, s, n)
        got, got_acc = run_matmul_dev(ctx, a, 1, k, qt)
        assert (got_acc == want_acc).all(), f"row {i}: i32 accumulators differ"
        finite = np.isfinite(want)
        assert (np.isfinite(got) == finite).all() and (bits(got[finite]) == bits(want[finite])).all(), f"row {i}: f32 outputs differ"
    # a row that does not start on a 16-byte boundary takes the two-launch path: same answer
    from peregrine_amd import _ffi
    a = rows[0]
    want, _ = orc.matmul_quantized(a, 1, k, q_t, s, n)
    shifted = DevBuf(ctx, host=np.concatenate([np.zeros(1, np.float32), a]))
    dout = DevBuf(ctx, n * 4)
    _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, C.c_void_p(shifted.ptr.value + 4), 1, k, qt._gpu, dout.ptr, None))
    ctx.sync()
    assert (bits(dout.to_host(np.float32)) == bits(want)).all()
    qt.free_gpu()


def test_matmul_quantized_extreme_integers(ctx, orc):
    # every product is (-127)*(-127) or 127*(-127): the largest accumulators the path can see
    from peregrine_amd import quant
    m, k, n = 70, 14336, 130
    say(f"matmul_quantized extremes m={m} k={k} n={n}")
    a = np.full((m, k), -3.0, np.float32)
    a[::2] = 3.0
    w = np.full((k, n), -0.5, np.float32)
    qt = quant.quantize_weights(w, k, n, ctx)
    got, acc = run_matmul_dev(ctx, a, m, k, qt)
    want_acc = np.where((np.arange(m) % 2 == 0)[:, None], -127 * 127 * k, 127 * 127 * k) * np.ones((1, n), np.int64)
    assert (acc.reshape(m, n) == want_acc).all()
    q, q_t, s = orc.quantize_weights(w, k, n)
    want, _ = orc.matmul_quantized(a, m, k, q_t, s, n)
    assert (bits(got) == bits(want)).all()


def test_matmul_quantized_shape_mismatch_is_an_error(ctx, orc):
    from peregrine_amd import quant, _ffi
    qt = quant.quantize_weights(np.ones(64 * 8, np.float32), 64, 8, ctx)
    with pytest.raises(ValueError):
        quant.matmul_quantized(np.zeros(2 * 32, np.float32), 2, 32, qt, ctx)  # assert_eq!(w.rows, k)
    qt.to_gpu(ctx)
    out = np.zeros(16, np.float32)
    st = _ffi.lib.pg_matmul_quantized(ctx.handle, C.c_void_p(out.ctypes.data), 2, 32, qt._gpu, C.c_void_p(out.ctypes.data))
    assert st == _ffi.PG_EINVAL and b"rows" in _ffi.lib.pg_last_error()
    assert quant.matmul_quantized(np.zeros(0, np.float32), 0, 64, qt, ctx).size == 0  # m = 0


def last_tile(ctx):
    """(rows, columns, K splits) of the most recent W8A8 matrix-core launch on this context."""
    from peregrine_amd import _ffi
    bm, bn, sp = C.c_int(), C.c_int(), C.c_int()
    _ffi.check(_ffi.lib.pg_gemm_w8a8_last_tile(ctx.handle, C.byref(bm), C.byref(bn), C.byref(sp)))
    return bm.value, bn.value, sp.value


def outlier_acts(orc, seed, m, k):
    """N(0,1) activations with 1 % of the channels scaled x20 (benchmark configuration 3)."""
    a = orc.rng_normal(seed, m * k).reshape(m, k)
    chan = np.random.default_rng(seed).choice(k, max(1, k // 100), replace=False)
    a[:, chan] *= 20
    return a


def np_epilogue(acc, a_s, w_s):
    """((acc as f32) * a_scale[m]) * w_scale[n] in IEEE single, the order of src/quant.rs:163."""
    return (acc.astype(np.float32) * a_s.astype(np.float32)[:, None]) * w_s.astype(np.float32)[None, :]


@pytest.mark.parametrize("m,k,n", [(700, 8200, 260), (412, 9001, 333), (300, 12000, 662), (257, 13990, 1031), (200, 9216, 402), (64, 13000, 300)])
def test_products_split_over_k_at_every_remainder_of_four_columns(ctx, orc, m, k, n):
    """K split over workgroups, up to 700 rows: the finishing launch by fours (with the accumulators and without), by single columns,
    and where the result lies one float off a multiple of four."""
    from peregrine_amd import quant, _ffi
    say(f"split over K m={m} k={k} n={n}")
    a = orc.rng_normal(4321 + m, m * k)
    qt = quant.quantize_weights(orc.rng_normal(8765 + n, k * n, 0.0, 0.02), k, n, ctx)
    got, got_acc = run_matmul_dev(ctx, a, m, k, qt)
    assert last_tile(ctx)[2] > 1
    rows = sorted({0, 63, m // 2, m - 2, m - 1})
    want, want_acc = orc.matmul_quantized(a.reshape(m, k)[rows].reshape(-1), len(rows), k, qt.data_i8_t, qt.scales, n)
    assert (got_acc.reshape(m, n)[rows].reshape(-1) == want_acc.reshape(-1)).all()
    assert (bits(got.reshape(m, n)[rows]).reshape(-1) == bits(want).reshape(-1)).all()
    x, y = DevBuf(ctx, host=a), DevBuf(ctx, (m * n + 1) * 4)
    for at in (0, 1):
        _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, x.ptr, m, k, qt._gpu, C.c_void_p(y.ptr.value + 4 * at), None))
        ctx.sync()
        assert (bits(y.to_host(np.float32)[at:at + m * n]) == bits(got.reshape(-1))).all()


# benchmark configuration 3: the seven products of one Llama-3-8B layer at M = 2048 are these four shapes;
# the last column is the output tile the dispatcher must pick (so a dispatcher change cannot
# silently leave a tile shape without a test)
PREFILL_SHAPES = [
    ("q/o_proj", 2048, 4096, 4096, (128, 256)),
    ("k/v_proj", 2048, 4096, 1024, (128, 64)),
    ("gate/up_proj", 2048, 4096, 14336, (256, 256)),
    ("down_proj", 2048, 14336, 4096, (128, 256)),
    ("unsplit 128x128", 1024, 1024, 4096, (128, 128)),
    ("two steps of K", 1024, 256, 4096, (128, 64)),
]


@pytest.mark.parametrize("name,m,k,n,tile", PREFILL_SHAPES, ids=[p[0] for p in PREFILL_SHAPES])
def test_prefill_shape_full_size_properties(ctx, orc, name, m, k, n, tile):
    """Every product shape of benchmark configuration 3 at full size (the oracle would need up to
    1.2e11 scalar MACs for one of them), checked through:
      (a) one row out of every 32-row band of the output (64 rows at M = 2048: every MFMA row tile
          of every workgroup tile, all columns) bit-exactly against the oracle, accumulators and f32;
      (b) 96 sampled columns over ALL rows against an int32 NumPy product of the oracle's
          quantised operands and the IEEE-single epilogue in the reference's order;
      (c) the sum over ALL accumulators against the exact identity
            sum_{m,n} acc[m,n] = sum_k (sum_m a_i8[m,k]) * (sum_n w_t[n,k])   (int64);
      (d) the f32-only call (no accumulator dump: the straight-line, non-temporal epilogue the
          benchmark runs) against the f32 output of the dumping call, every element;
      (e) the tile shape the dispatcher chose."""
    from peregrine_amd import quant, _ffi
    say(f"prefill full size {name}: m={m} k={k} n={n}")
    a = outlier_acts(orc, 4321 + n, m, k)
    w = orc.rng_normal(8765 + k, k * n, 0.0, 0.02)
    q, q_t, s = orc.quantize_weights(w, k, n)
    qt = quant.QuantizedTensor(q, q_t, s, k, n)
    del w
    got, acc = run_matmul_dev(ctx, a, m, k, qt)
    assert last_tile(ctx) == tile + (1,), f"dispatcher picked {last_tile(ctx)}, the test expects {tile}"
    got, acc = got.reshape(m, n), acc.reshape(m, n)
    a_i8, a_s = orc.quantize_activations(a, m, k)
    a_i8 = a_i8.reshape(m, k)
    # (c)
    col = a_i8.astype(np.int64).sum(axis=0)
    wsum = q_t.reshape(n, k).astype(np.int64).sum(axis=0)
    assert int(acc.astype(np.int64).sum()) == int((col * wsum).sum())
    # (a)
    rng = np.random.default_rng(2)
    rows = np.arange(0, m, 32) + rng.integers(0, 32, size=(m + 31) // 32)
    rows = rows[rows < m]
    want, want_acc = orc.matmul_quantized(a[rows], len(rows), k, q_t, s, n)
    assert (acc[rows] == want_acc.reshape(len(rows), n)).all()
    assert (bits(got[rows]) == bits(want.reshape(len(rows), n))).all()
    # (b)
    cols = np.unique(np.concatenate([rng.choice(n, 90, replace=False), [0, 31, 32, n - 33, n - 32, n - 1]]))
    wc = q_t.reshape(n, k)[cols].astype(np.float64)          # [cols, k]
    acc_c = (a_i8.astype(np.float64) @ wc.T).astype(np.int32)  # exact: every partial sum is an integer below 2^53
    assert (acc[:, cols] == acc_c).all()
    assert (bits(got[:, cols]) == bits(np_epilogue(acc_c, a_s, s[cols]))).all()
    # (d)
    da = DevBuf(ctx, host=a)
    dout = DevBuf(ctx, m * n * 4)
    _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr, None))
    ctx.sync()
    assert last_tile(ctx) == tile + (1,)
    assert (bits(dout.to_host(np.float32)) == bits(got).reshape(-1)).all(), "f32-only epilogue differs"
    qt.free_gpu()


# pg_gemm_w8a8_force_tile codes -> output tile
TILES = {1: (64, 64), 2: (256, 256), 3: (128, 256), 4: (128, 64), 5: (128, 128)}


@pytest.mark.parametrize("m,k,n", [(300, 512, 1000), (512, 384, 768), (70, 128, 257)])
def test_every_gemm_tile_gives_the_same_bits(ctx, orc, m, k, n):
    """Each instantiation of the matrix-core kernel, forced in turn on ragged and whole-tile
    shapes, with and without the accumulator dump, against the oracle."""
    from peregrine_amd import quant, _ffi
    a = outlier_acts(orc, 99 + m, m, k)
    w = orc.rng_normal(55 + n, k * n, 0.0, 0.02)
    q, q_t, s = orc.quantize_weights(w, k, n)
    qt = quant.QuantizedTensor(q, q_t, s, k, n).to_gpu(ctx)
    want, want_acc = orc.matmul_quantized(a, m, k, q_t, s, n)
    da = DevBuf(ctx, host=a)
    dout, dacc = DevBuf(ctx, m * n * 4), DevBuf(ctx, m * n * 4)
    try:
        for code, tile in TILES.items():
            say(f"gemm tile {tile} on m={m} k={k} n={n}")
            _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, code))
            for acc_ptr in (dacc.ptr, None):
                _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr, acc_ptr))
                ctx.sync()
                bm, bn, sp = last_tile(ctx)
                if sp == 1:  # (a split product keeps its own row tile)
                    assert (bm, bn) == tile
                assert (bits(dout.to_host(np.float32)) == bits(want)).all(), f"tile {tile}: f32 outputs differ"
            assert (dacc.to_host(np.int32) == want_acc).all(), f"tile {tile}: accumulators differ"
    finally:
        _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, 0))
    assert _ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, 9) == _ffi.PG_EINVAL
    qt.free_gpu()


@pytest.mark.parametrize("m,k,n", [(257, 128, 510),       # panels of 192 columns that end behind the weight's padding; one step of K
                                    (512, 300, 768), (90, 700, 193), (300, 640, 1030)])
def test_wide_gemm_tiles_give_the_same_bits(ctx, orc, m, k, n):
    """The tiles of codes 6 to 8, and 64x64, as the others above (from 33 rows on a tile that is asked for is what runs)."""
    from peregrine_amd import quant, _ffi
    a = outlier_acts(orc, 17 + m, m, k)
    w = orc.rng_normal(18 + n, k * n, 0.0, 0.02)
    q, q_t, s = orc.quantize_weights(w, k, n)
    qt = quant.QuantizedTensor(q, q_t, s, k, n).to_gpu(ctx)
    want, want_acc = orc.matmul_quantized(a, m, k, q_t, s, n)
    da = DevBuf(ctx, host=a)
    dout, dacc = DevBuf(ctx, m * n * 4 + 4), DevBuf(ctx, m * n * 4)
    try:
        for code, tile in {6: (128, 192), 7: (256, 128), 8: (256, 192), 1: (64, 64)}.items():
            say(f"gemm tile {tile} on m={m} k={k} n={n}")
            _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, code))
            for acc_ptr, skew in ((dacc.ptr, 0), (None, 0), (None, 4)):   # an output off the lines is stored plainly
                out = C.c_void_p(dout.ptr.value + skew)
                _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, out, acc_ptr))
                ctx.sync()
                bm, bn, sp = last_tile(ctx)
                assert sp == 1 and (bm, bn) == tile
                got = dout.to_host(np.float32)[skew // 4:skew // 4 + m * n]
                assert (bits(got) == bits(want)).all(), f"tile {tile}: f32 outputs differ"
            assert (dacc.to_host(np.int32) == want_acc).all(), f"tile {tile}: accumulators differ"
    finally:
        _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, 0))
    qt.free_gpu()


@pytest.mark.parametrize("m,k,n,tile", [(400, 1024, 4096, None), (2100, 640, 2000, None), (1600, 4100, 3300, None), (1200, 9000, 4100, None),
                                         (1400, 4000, 2000, None), (1024, 512, 3968, (128, 128)), (600, 3744, 10144, None)])
def test_chosen_gemm_tiles_against_numpy(ctx, orc, m, k, n, tile):
    """Products whose kernel the estimates choose, exact integers against an int64 product."""
    from peregrine_amd import quant, _ffi
    rng = np.random.default_rng(m)
    a = rng.integers(-127, 128, (m, k)).astype(np.float32)
    a[:, 0] = 127.0                                        # so that the row scale is 1
    qi = rng.integers(-127, 128, (k, n)).astype(np.int8)
    qt = quant.QuantizedTensor(qi.reshape(-1), np.ascontiguousarray(qi.T).reshape(-1), np.ones(n, np.float32), k, n).to_gpu(ctx)
    da, dout = DevBuf(ctx, host=a), DevBuf(ctx, m * n * 4)
    _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr, None))
    ctx.sync()
    say(f"gemm m={m} k={k} n={n} ran {last_tile(ctx)}")
    assert tile is None or last_tile(ctx)[:2] == tile
    got = dout.to_host(np.float32).reshape(m, n)
    want = (a.astype(np.float64) @ qi.astype(np.float64)).astype(np.float32)   # |sum| < 2^53; rounded once, as (float)acc is
    assert (bits(got) == bits(want)).all()
    qt.free_gpu()


@pytest.mark.parametrize("m,k,n,kernel", H.INT8_ROUTES)
def test_int8_routes_against_numpy(ctx, orc, m, k, n, kernel):
    """The same on ragged products of every kernel from 33 rows on (test_host_runtime.py says that these kernels run), with the
    accumulators."""
    from peregrine_amd import quant, _ffi
    say(f"int8 route m={m} k={k} n={n} {kernel}")
    rng = np.random.default_rng(m + k)
    a = rng.integers(-127, 128, (m, k)).astype(np.float32)
    a[:, 0] = 127.0
    qi = rng.integers(-127, 128, (k, n)).astype(np.int8)
    qt = quant.QuantizedTensor(qi.reshape(-1), np.ascontiguousarray(qi.T).reshape(-1), np.ones(n, np.float32), k, n).to_gpu(ctx)
    da, dout, dacc = DevBuf(ctx, host=a), DevBuf(ctx, m * n * 4), DevBuf(ctx, m * n * 4)
    want = a.astype(np.float64) @ qi.astype(np.float64)
    for acc in (None, dacc.ptr):
        _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr, acc))
        assert (bits(dout.to_host(np.float32).reshape(m, n)) == bits(want.astype(np.float32))).all()
    assert (dacc.to_host(np.int32).reshape(m, n) == want).all()
    qt.free_gpu()


@pytest.mark.parametrize("semantics,m,k,n", [("w8a8", 1024, 96, 12800), ("w8a8", 1005, 96, 12770), ("w8a8", 1009, 160, 12799), ("w8a32", 1024, 96, 11520),
                                             ("w8a32", 1005, 96, 11390), ("w8a32", 385, 100, 600), ("w8a32", 384, 96, 640)])
def test_int8_tiles_store_whole_and_cut_tiles(ctx, orc, semantics, m, k, n):
    """Products of more than a tile either way, with and without cut tiles and rows that begin on a line: the f32 output, the accumulators,
    both, and W8A32 in one launch and over two planes of accumulators.  Small integers: every result is exact."""
    from peregrine_amd import quant, _ffi
    say(f"int8 tiles {semantics} m={m} k={k} n={n}")
    rng = np.random.default_rng(m + n)
    a = rng.integers(-127, 128, (m, k)).astype(np.float32)
    a[:, 0] = 127.0                                        # so that W8A8's row scale is 1
    qi = rng.integers(-127, 128, (k, n)).astype(np.int8)
    qt = quant.QuantizedTensor(qi.reshape(-1), np.ascontiguousarray(qi.T).reshape(-1), np.ones(n, np.float32), k, n).to_gpu(ctx)
    want = a @ qi.astype(np.float32)                       # |sums| < 2^24: exact in any order
    da, dout, dacc = DevBuf(ctx, host=a), DevBuf(ctx, m * n * 4), DevBuf(ctx, m * n * 4)
    if semantics == "w8a32":
        _ffi.check(_ffi.lib.pg_matmul_dequant_i8_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr))
        assert (dout.to_host(np.float32).reshape(m, n) == want).all()
    else:
        for acc in (None, dacc.ptr):
            _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr, acc))
            assert (dout.to_host(np.float32).reshape(m, n) == want).all()
        assert (dacc.to_host(np.int32).reshape(m, n) == want.astype(np.int32)).all()
    qt.free_gpu()


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6, 7, 8, "w8a32"])
@pytest.mark.parametrize("m,n", [(4300, 2690), (1030, 5000), (3221, 300)])
def test_int8_tiles_in_strips(ctx, tile, m, n):
    """Every tile shape over more row tiles than a strip holds, the last strip shorter (1030 rows: with and without strips): each tile is made
    once, where it belongs.  Small integers: every result is exact."""
    from peregrine_amd import quant, _ffi
    say(f"int8 tiles in strips {tile} m={m} n={n}")
    k = 70
    rng = np.random.default_rng(m)
    a = rng.integers(-127, 128, (m, k)).astype(np.float32)
    a[:, 0] = 127.0                                        # so that W8A8's row scale is 1
    qi = rng.integers(-127, 128, (k, n)).astype(np.int8)
    qt = quant.QuantizedTensor(qi.reshape(-1), np.ascontiguousarray(qi.T).reshape(-1), np.ones(n, np.float32), k, n).to_gpu(ctx)
    da, dout = DevBuf(ctx, host=a), DevBuf(ctx, m * n * 4)
    if tile == "w8a32":
        _ffi.check(_ffi.lib.pg_matmul_dequant_i8_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr))
    else:
        _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, tile))
        try:
            _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, dout.ptr, None))
        finally:
            _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, 0))
    assert (dout.to_host(np.float32).reshape(m, n) == a @ qi.astype(np.float32)).all()   # |sums| < 2^24: exact in any order
    row_tiles, strip = C.c_int(), C.c_int()
    _ffi.check(_ffi.lib.pg_gemm_w8a8_last_order(ctx.handle, C.byref(row_tiles), C.byref(strip)))
    if m > 1030:
        assert strip.value < row_tiles.value and (tile == "w8a32" or row_tiles.value % strip.value), (row_tiles.value, strip.value)
    qt.free_gpu()


def run_multi(ctx, da, m, k, qts, douts):
    from peregrine_amd import _ffi
    wtab = (C.c_void_p * len(qts))(*[q._gpu.value for q in qts])
    otab = (C.c_void_p * len(qts))(*[d.ptr.value for d in douts])
    _ffi.check(_ffi.lib.pg_matmul_quantized_multi_dev(ctx.handle, da.ptr, m, k, wtab, len(qts), otab))
    ctx.sync()


@pytest.mark.parametrize("m,k,ns", [(300, 512, (1000, 130, 257)), (257, 128, (64, 64, 64, 64)), (40, 1024, (300, 77)),
                                     (1, 4096, (1024, 512)), (1, 14336, (300, 77, 4096)), (3, 200, (33,)), (2048, 4096, (4096, 1024, 1024)),
                                     (2048, 4096, (14336, 14336)), (8, 4096, (4096, 1024, 1030)), (32, 1000, (8200, 520)),
                                     (1, 4096, (14336, 14336))],
                         ids=["ragged3", "four", "few-rows", "one-row", "one-row-long-k", "single", "qkv", "gate-up",
                              "qkv-8-rows-quantised-once", "32-rows-quantised-once", "one-row-gate-up-as-the-decode-benchmark-runs-it"])
def test_matmul_quantized_multi_equals_the_single_products(ctx, orc, m, k, ns):
    """Several weights against one activation matrix (the reference's fused QKV / gate|up
    products): every output equals the single product bit for bit, and sampled rows equal the
    oracle."""
    from peregrine_amd import quant, _ffi
    say(f"matmul_quantized_multi m={m} k={k} ns={ns}")
    a = outlier_acts(orc, 7 + m, m, k)
    da = DevBuf(ctx, host=a)
    qts, parts = [], []
    for i, n in enumerate(ns):
        w = orc.rng_normal(100 + 13 * i + n, k * n, 0.0, 0.02)
        q, q_t, s = orc.quantize_weights(w, k, n)
        parts.append((q_t, s))
        qts.append(quant.QuantizedTensor(q, q_t, s, k, n).to_gpu(ctx))
    douts = [DevBuf(ctx, m * n * 4) for n in ns]
    run_multi(ctx, da, m, k, qts, douts)
    if m == 2048:
        assert last_tile(ctx)[:2] == (256, 256)  # gate, up: a launch each; q|k|v: one launch of 192 tiles
    rows = np.unique(np.random.default_rng(3).choice(m, min(m, 24), replace=False))
    single = DevBuf(ctx, m * max(ns) * 4)
    for i, n in enumerate(ns):
        got = douts[i].to_host(np.float32)
        _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qts[i]._gpu, single.ptr, None))
        ctx.sync()
        assert (bits(got) == bits(single.to_host(np.float32, m * n))).all(), f"weight {i}: differs from the single product"
        want, _ = orc.matmul_quantized(a[rows], len(rows), k, parts[i][0], parts[i][1], n)
        assert (bits(got.reshape(m, n)[rows]) == bits(want.reshape(len(rows), n))).all(), f"weight {i}: differs from the oracle"
    # argument errors: too many weights, a weight with another k
    five = (C.c_void_p * 5)(*[qts[0]._gpu.value] * 5)
    outs5 = (C.c_void_p * 5)(*[douts[0].ptr.value] * 5)
    assert _ffi.lib.pg_matmul_quantized_multi_dev(ctx.handle, da.ptr, m, k, five, 5, outs5) == _ffi.PG_EINVAL
    assert _ffi.lib.pg_matmul_quantized_multi_dev(ctx.handle, da.ptr, m, k + 1, five, 1, outs5) == _ffi.PG_EINVAL
    for qt in qts:
        qt.free_gpu()


def test_wire_record_straight_to_device(ctx, orc):
    """read_quantized_tensor + to_gpu in one call (reference src/serial.rs:161-222,
    src/quant.rs:174-181): the device tensor multiplies exactly like the original."""
    import io
    import ctypes as C
    from peregrine_amd import serial, _ffi
    from peregrine_amd.quant import QuantizedTensor
    say("wire record -> device tensor")
    rows, cols, m = 96, 40, 3
    w = orc.rng_normal(31, rows * cols, 0.0, 0.02)
    q, q_t, s = orc.quantize_weights(w, rows, cols)
    buf = io.BytesIO()
    serial.write_quantized_tensor(buf, "odd", QuantizedTensor(q, q_t, s, rows, cols))  # 3-byte name: unaligned payload
    h, used = serial.quantized_tensor_to_gpu(buf.getvalue() + b"trailing", ctx)
    assert used == len(buf.getvalue())
    a = orc.rng_normal(32, m * rows)
    out = np.empty(m * cols, np.float32)
    _ffi.check(_ffi.lib.pg_matmul_quantized(ctx.handle, C.c_void_p(a.ctypes.data), m, rows, h, C.c_void_p(out.ctypes.data)))
    want, _ = orc.matmul_quantized(a, m, rows, q_t, s, cols)
    assert (out.view(np.uint32) == want.view(np.uint32)).all()
    _ffi.lib.pg_qtensor_free(ctx.handle, h)


W8A32_SHAPES = [(32, 128, 64), (1, 4096, 1024), (3, 200, 77), (70, 4096, 300), (191, 256, 130),
                (192, 512, 300), (256, 384, 256), (300, 1000, 520), (700, 256, 1000)]


@pytest.mark.parametrize("m,k,n", W8A32_SHAPES)
def test_matmul_dequant_i8_vs_oracle(ctx, orc, m, k, n):
    """W8A32, the reference's GPU numerics (src/metal/shaders.rs:2329-2375).  Two bars: against
    the exact (float64) product of the same f32 activations and dequantised weights, 1e-5 of
    max(|ref|, rms(ref)) -- this implementation's own error (23/24-bit fixed point per row, so a
    row with x20 outlier channels loses ~6 bits on its ordinary elements; exact integer sums);
    against the oracle's K-sequential f32 sum, 2e-5 -- at K = 4096 that sum itself carries up to
    ~1e-5 of rounding error."""
    from peregrine_amd import quant
    say(f"matmul_dequant_i8 m={m} k={k} n={n}")
    a = orc.rng_normal(11 + m, m * k)
    a.reshape(m, k)[:, :: max(1, k // 37)] *= 20
    w = orc.rng_normal(12 + n, k * n, 0.0, 0.02)
    q, q_t, s = orc.quantize_weights(w, k, n)
    qt = quant.QuantizedTensor(q, q_t, s, k, n)
    got = quant.matmul_dequant_i8(a, m, k, qt, ctx).reshape(m, n)
    want = orc.matmul_dequant_i8(a, m, k, q, s, n).reshape(m, n)
    exact = a.reshape(m, k).astype(np.float64) @ orc.dequantize(q, s, k, n).reshape(k, n).astype(np.float64)
    for r in range(m):
        H.assert_close_rel(got[r], exact[r], 1e-5, f"row {r} vs exact")
        H.assert_close_rel(got[r], want[r], 2e-5, f"row {r} vs f32 oracle")
    qt.free_gpu()


@pytest.mark.parametrize("m,k,n,runs", [(587, 4137, 316, 9), (670, 8232, 281, 9)])
def test_products_split_over_k_whose_last_run_is_one_tile_of_k(ctx, orc, m, k, n, runs):
    """33 k-tiles in runs of four, 65 in runs of eight."""
    from peregrine_amd import quant
    say(f"split over K, a last run of one k-tile, m={m} k={k} n={n}")
    a = orc.rng_normal(99 + m, m * k)
    qt = quant.quantize_weights(orc.rng_normal(98 + n, k * n, 0.0, 0.02), k, n, ctx)
    got, got_acc = run_matmul_dev(ctx, a, m, k, qt)
    assert last_tile(ctx) == (64, 64, runs)
    rows = sorted({0, 63, m // 2, m - 1})
    want, want_acc = orc.matmul_quantized(a.reshape(m, k)[rows].reshape(-1), len(rows), k, qt.data_i8_t, qt.scales, n)
    assert (got_acc.reshape(m, n)[rows].reshape(-1) == want_acc.reshape(-1)).all()
    assert (bits(got.reshape(m, n)[rows]).reshape(-1) == bits(want).reshape(-1)).all()


@pytest.mark.parametrize("m,k,n,runs", [(286, 7055, 832, 3), (768, 8136, 111, 8), (57, 10391, 3087, 4), (485, 7086, 294, 6), (164, 9108, 1114, 4), (330, 12000, 130, 8), (33, 132000, 7, 8)])
def test_matmul_dequant_i8_split_over_k(ctx, orc, m, k, n, runs):
    """K in runs over workgroups: whole numbers as activations and powers of two as scales make the product exact, in even and odd
    numbers of columns, and where the result lies one float off a multiple of two."""
    from peregrine_amd import quant, _ffi
    say(f"matmul_dequant_i8 split over K m={m} k={k} n={n}")
    rng = np.random.default_rng(m + n)
    a = rng.integers(-100, 101, size=(m, k)).astype(np.float32)
    q = rng.integers(-127, 128, size=(k, n), dtype=np.int8)
    s = (2.0 ** rng.integers(-12, -4, size=n)).astype(np.float32)
    qt = quant.QuantizedTensor(q.reshape(-1), np.ascontiguousarray(q.T).reshape(-1), s, k, n)
    qt.to_gpu(ctx)
    rows = sorted({0, 63, 64, m // 2, m - 1} & set(range(m)))
    want = ((a[rows].astype(np.int64) @ q.astype(np.int64)).astype(np.float64) * s).astype(np.float32)
    x, y = DevBuf(ctx, host=a), DevBuf(ctx, (m * n + 1) * 4)
    for at in (0, 1):
        _ffi.check(_ffi.lib.pg_matmul_dequant_i8_dev(ctx.handle, x.ptr, m, k, qt._gpu, C.c_void_p(y.ptr.value + 4 * at)))
        ctx.sync()
        assert last_tile(ctx) == (64, 64, runs)
        got = y.to_host(np.float32)[at:at + m * n].reshape(m, n)[rows]
        assert (got == want).all()
    qt.free_gpu()


@pytest.mark.parametrize("m,k,n,runs", [(286, 7055, 832, 3), (768, 7200, 111, 8), (57, 10391, 3087, 4), (164, 9108, 1114, 4), (33, 20000, 7, 8)])
def test_matmul_dequant_i8_split_over_k_rounds_once(ctx, orc, m, k, n, runs):
    """Ordinary rows, of a small and of a large scale, of infinities and of NaN: K in runs (the last of 768 x 7200 a single k-tile) gives the bits of the whole
    product, which a tile override makes in another way."""
    from peregrine_amd import quant, _ffi
    say(f"matmul_dequant_i8 split against whole m={m} k={k} n={n}")
    rng = np.random.default_rng(m + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::53] *= 20.0
    a[1] *= np.float32(1e-30)
    a[2] *= np.float32(1e30)
    a[3, k // 2], a[4, 0] = np.inf, np.nan
    qt = quant.quantize_weights(orc.rng_normal(77 + n, k * n, 0.0, 0.02), k, n, ctx)
    qt.to_gpu(ctx)
    x, y = DevBuf(ctx, host=a), DevBuf(ctx, m * n * 4)
    got = []
    for tile in (0, 1):
        _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, tile))
        try:
            _ffi.check(_ffi.lib.pg_matmul_dequant_i8_dev(ctx.handle, x.ptr, m, k, qt._gpu, y.ptr))
            ctx.sync()
        finally:
            _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, 0))
        assert last_tile(ctx)[2] == (1 if tile else runs)
        got.append(y.to_host(np.float32).copy().reshape(m, n))
    same = (bits(got[0]) == bits(got[1])).reshape(m, n) | (np.isnan(got[0]) & np.isnan(got[1]))
    assert same.all(), np.argwhere(~same)[:5]
    assert np.isfinite(got[0][5:]).all() and (np.abs(got[0][5:]).max(axis=1) > 0).all()
    exact = a[5:].astype(np.float64) @ orc.dequantize(qt.data_i8, qt.scales, k, n).reshape(k, n).astype(np.float64)
    for r in (0, m // 2, m - 6):
        H.assert_close_rel(got[0][5 + r], exact[r], 1e-5, f"row {5 + r} vs exact")
    qt.free_gpu()


def test_matmul_dequant_i8_combining_epilogue_on_every_tile(ctx, orc):
    """Where the planes are stacked (beyond one launch's offsets; under a tile override) the product of the plane of weight
    65536 finishes the sum in its epilogue (it reads the other two planes' accumulators).  Every tile shape of the matrix-core
    kernel in turn, on a ragged shape (the bounds-checked epilogue at the edges, the straight-line one inside), and two
    shapes of many 256x256 tiles (whole tiles only, and ragged): exact small integers in, exact integers out, and
    the float64 product as the bar for random data."""
    from peregrine_amd import quant, _ffi
    for m, k, n, force in [(300, 256, 520, c) for c in TILES] + [(2048, 128, 5888, 2), (2050, 128, 5900, 2)]:
        say(f"matmul_dequant_i8 m={m} k={k} n={n} tile override {force}")
        a = orc.rng_normal(21 + m, m * k)
        a.reshape(m, k)[:, :: max(1, k // 37)] *= 20
        w = orc.rng_normal(22 + n, k * n, 0.0, 0.02)
        q, q_t, s = orc.quantize_weights(w, k, n)
        qt = quant.QuantizedTensor(q, q_t, s, k, n)
        ai = (np.arange(m * k, dtype=np.float32) % 9 - 4).reshape(m, k)
        qi = (np.arange(k * n).reshape(k, n) % 13 - 6).astype(np.int8)
        qt_int = quant.QuantizedTensor(qi.reshape(-1), np.ascontiguousarray(qi.T).reshape(-1), np.ones(n, np.float32), k, n)
        try:
            _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, force))
            got = quant.matmul_dequant_i8(a, m, k, qt, ctx).reshape(m, n)
            assert last_tile(ctx)[:2] == TILES[force]
            got_int = quant.matmul_dequant_i8(ai, m, k, qt_int, ctx).reshape(m, n)
        finally:
            _ffi.check(_ffi.lib.pg_gemm_w8a8_force_tile(ctx.handle, 0))
        assert (got_int == (ai.astype(np.int64) @ qi.astype(np.int64))).all(), "integer inputs: the product is not exact"
        exact = a.reshape(m, k).astype(np.float64) @ orc.dequantize(q, s, k, n).reshape(k, n).astype(np.float64)
        for r in range(m):
            H.assert_close_rel(got[r], exact[r], 1e-5, f"row {r} vs exact")
        qt.free_gpu()
        qt_int.free_gpu()


def test_matmul_dequant_i8_reference_tolerance_and_closed_form(ctx, orc):
    """tests/quant_parity.rs:79-146 restated: the W8A32 result is within 10 % / 0.02 of the f32
    product of the unquantised weights; plus integer inputs with unit scales give exact integers,
    zero rows give zeros and a NaN poisons exactly its row."""
    from peregrine_amd import quant
    m, k, n = 32, 128, 64
    a = H.mod_pattern(m * k, 7, 3, 200, 200, 0.5)
    w = H.mod_pattern(k * n, 13, 7, 200, 200, 0.5)
    qt = quant.quantize_weights(w, k, n, ctx)
    got = quant.matmul_dequant_i8(a, m, k, qt, ctx)
    ref = orc.matmul_f32(a, w, m, k, n)
    diff = np.abs(got - ref)
    assert ((diff / np.maximum(np.abs(ref), 1e-6) < 0.10) | (diff < 0.02)).all()
    ai = (np.arange(m * k, dtype=np.float32) % 9 - 4).reshape(m, k)
    ai[3] = 0
    qi = (np.arange(k * n).reshape(k, n) % 13 - 6).astype(np.int8)
    qt2 = quant.QuantizedTensor(qi.reshape(-1), np.ascontiguousarray(qi.T).reshape(-1), np.ones(n, np.float32), k, n)
    got = quant.matmul_dequant_i8(ai, m, k, qt2, ctx).reshape(m, n)
    assert (got == ai.astype(np.int64) @ qi.astype(np.int64)).all() and (got[3] == 0).all()
    ai[5, 17] = np.nan
    got = quant.matmul_dequant_i8(ai, m, k, qt2, ctx).reshape(m, n)
    assert np.isnan(got[5]).all() and np.isfinite(np.delete(got, 5, axis=0)).all()
    with pytest.raises(ValueError):
        quant.matmul_dequant_i8(ai, m, k + 1, qt2, ctx)


@pytest.mark.parametrize("m,k,n", [
    (1, 32, 1), (3, 7, 5), (64, 64, 64), (63, 33, 65), (17, 96, 241),   # one word out; 16 KB, 4 bytes less, 4 bytes more
    (512, 512, 40), (511, 513, 40), (1025, 257, 40),                    # 1 MB in, just below, just above (two pieces)
    (1024, 64, 1024), (1025, 64, 1023), (1537, 64, 2049), (2050, 1100, 1030),  # one window of 4 MB out, 4 bytes less, several; 9 MB in
])
def test_host_arrays_cross_whole(ctx, m, k, n):
    """The host-array call against the device-pointer call, bit for bit, at the edges of the transfers' pieces; twice,
    so that the second finds the first one's words in the staging memory."""
    from peregrine_amd import quant, _ffi
    say(f"host arrays m={m} k={k} n={n}")
    rng = np.random.default_rng(m + n)
    qt = quant.quantize_weights(rng.standard_normal(k * n).astype(np.float32), k, n, ctx).to_gpu(ctx)
    for _ in range(2):
        a = rng.standard_normal(m * k).astype(np.float32)
        da, do = DevBuf(ctx, host=a), DevBuf(ctx, nbytes=4 * m * n)
        _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, da.ptr, m, k, qt._gpu, do.ptr, None))
        ctx.sync()
        want = do.to_host(np.float32)
        got = quant.matmul_quantized(a, m, k, qt, ctx)
        assert (got.view(np.uint32) == want.view(np.uint32)).all()


@pytest.mark.parametrize("m,k,n", [
    (2, 128, 16), (16, 4096, 1000), (16, 640, 33), (17, 1000, 250), (32, 4096, 600),     # the few-row kernel: three and six tiles of planes
    (33, 128, 64), (64, 700, 65), (65, 4000, 300), (197, 1024, 515), (129, 256, 4097),   # 64x64 tiles, ragged
    (1030, 384, 3600), (1100, 130, 3333),                                                # 128x128 tiles, ragged
])
def test_matmul_dequant_i8_one_launch(ctx, orc, m, k, n):
    """W8A32 over three digit planes in one launch at the edges of its kernels' tiles: exact small integers in, exact
    integers out, and the float64 product as the bar for random data."""
    from peregrine_amd import quant
    say(f"matmul_dequant_i8 one launch m={m} k={k} n={n}")
    ai = (np.arange(m * k, dtype=np.float32) % 9 - 4).reshape(m, k)
    qi = (np.arange(k * n).reshape(k, n) % 13 - 6).astype(np.int8)
    qt = quant.QuantizedTensor(qi.reshape(-1), None, np.ones(n, np.float32), k, n)
    got = quant.matmul_dequant_i8(ai, m, k, qt, ctx).reshape(m, n)
    assert (got == ai @ qi.astype(np.float32)).all(), "integer inputs: the product is not exact"
    qt.free_gpu()
    a = orc.rng_normal(41 + m, m * k)
    a.reshape(m, k)[:, :: max(1, k // 37)] *= 20
    q, q_t, s = orc.quantize_weights(orc.rng_normal(42 + n, k * n, 0.0, 0.02), k, n)
    qt = quant.QuantizedTensor(q, q_t, s, k, n)
    got = quant.matmul_dequant_i8(a, m, k, qt, ctx).reshape(m, n)
    exact = a.reshape(m, k).astype(np.float64) @ orc.dequantize(q, s, k, n).reshape(k, n).astype(np.float64)
    for r in range(m):
        H.assert_close_rel(got[r], exact[r], 1e-5, f"row {r} vs exact")
    qt.free_gpu()


@pytest.mark.parametrize("m,k,n", [
    (519, 2221, 73), (186, 408, 2870), (211, 102, 3608), (1060, 665, 1904), (770, 105, 2959), (526, 1666, 3890),   # the tiles
    (391, 631, 2419), (580, 209, 3254), (1071, 1731, 3635),
    (124, 1073, 515), (512, 174, 73), (212, 174, 73), (74, 396, 1118), (33, 128, 17), (513, 1000, 64),             # groups of rows, their ends
    (9, 1530, 4100), (8, 3000, 70), (17, 1500, 30), (32, 1409, 2049), (31, 2500, 4097),                             # few rows of long K
] + [r[:3] for r in H.W8A32_ROUTES])
def test_matmul_dequant_i8_on_every_kernel(ctx, orc, m, k, n):
    """Each kernel of the one launch from 33 rows on, at ragged sizes (the last ones: test_host_runtime.py says which runs).  Small integers are exact; random
    rows are within the activation step (2^-23 of the row's largest value a value) and one rounding of the float64 product."""
    from peregrine_amd import quant
    say(f"matmul_dequant_i8 kernels m={m} k={k} n={n}")
    rng = np.random.default_rng(m + k)
    qi = rng.integers(-127, 128, (k, n)).astype(np.int8)
    s = rng.uniform(0.5e-3, 2e-3, n).astype(np.float32)
    ones = quant.QuantizedTensor(qi.reshape(-1), np.ascontiguousarray(qi.T).reshape(-1), np.ones(n, np.float32), k, n)
    ai = rng.integers(-9, 10, (m, k)).astype(np.float32)
    got = quant.matmul_dequant_i8(ai, m, k, ones, ctx).reshape(m, n)
    assert (got == (ai.astype(np.float64) @ qi.astype(np.float64))).all()
    qt = quant.QuantizedTensor(qi.reshape(-1), np.ascontiguousarray(qi.T).reshape(-1), s, k, n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    got = quant.matmul_dequant_i8(a, m, k, qt, ctx).reshape(m, n).astype(np.float64)
    w = qi.astype(np.float64) * s.astype(np.float64)
    want = a.astype(np.float64) @ w
    bound = np.abs(a).max(1, keepdims=True) * 2.0 ** -23 * np.abs(w).sum(0, keepdims=True) + np.abs(want) * 2.0 ** -23
    assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("m,k,n", [(1, 256, 50257), (32, 384, 65536), (33, 130, 128256), (191, 256, 50257), (383, 128, 45825),
                                   (192, 256, 50257)])
def test_matmul_dequant_i8_wide_weights(ctx, m, k, n):
    """W8A32 over a vocabulary's columns: exact small integers in, exact integers out, on rows and columns of every tile's
    beginning and end; and the float64 product there for random data."""
    from peregrine_amd import quant
    say(f"matmul_dequant_i8 wide weights m={m} k={k} n={n}")
    rng = np.random.default_rng(m + n)
    rows = np.unique(np.r_[0, m // 2, m - 1, rng.integers(0, m, 5)])
    cols = np.unique(np.r_[0:40, n // 2, n - 300 : n, rng.integers(0, n, 300)])
    ai = (np.arange(m * k, dtype=np.float32) % 9 - 4).reshape(m, k)
    qi = rng.integers(-127, 128, (k, n), dtype=np.int8)
    qt = quant.QuantizedTensor(qi.reshape(-1), None, np.ones(n, np.float32), k, n)
    got = quant.matmul_dequant_i8(ai, m, k, qt, ctx).reshape(m, n)
    w = qi[:, cols].astype(np.float64)
    assert (got[np.ix_(rows, cols)] == ai[rows].astype(np.float64) @ w).all(), "integer inputs: the product is not exact"
    a = rng.standard_normal((m, k)).astype(np.float32)
    got = quant.matmul_dequant_i8(a, m, k, qt, ctx).reshape(m, n)
    exact = a[rows].astype(np.float64) @ w
    for i, r in enumerate(rows):
        H.assert_close_rel(got[r, cols], exact[i], 1e-5, f"row {r} vs exact")
    assert np.isfinite(got).all() and (np.abs(got).max(axis=1) > 0).all()
    qt.free_gpu()


@pytest.mark.parametrize("rows,cols", [(3, 4), (2, 5), (5, 1023), (4, 1025), (6, 4098), (2, 4099), (700, 4097),
                                       (2, 16381), (600, 16389), (1, 32767), (1, 32772), (3, 3)])
def test_row_kernels_on_rows_of_any_length(ctx, orc, rows, cols):
    """The row kernels at the edges of their workgroups (256 and 1024 threads) and register counts, with one to three
    columns past the last whole vector: int8 rows bit for bit through a product (padded rows), and the digit rows of
    W8A32 through exact integers."""
    from peregrine_amd import quant
    say(f"row kernels rows={rows} cols={cols}")
    n = 3
    a = orc.rng_normal(51 + cols, rows * cols).reshape(rows, cols)
    a[-1, -1] = 40.0
    q, q_t, s = orc.quantize_weights(orc.rng_normal(52 + cols, cols * n, 0.0, 0.02), cols, n)
    qt = quant.QuantizedTensor(q, q_t, s, cols, n)
    got = quant.matmul_quantized(a, rows, cols, qt, ctx)
    want, _ = orc.matmul_quantized(a, rows, cols, q_t, s, n)
    assert (bits(got) == bits(want)).all()
    ai = (np.arange(rows * cols, dtype=np.float32) % 9 - 4).reshape(rows, cols)
    qi = (np.arange(cols * n).reshape(cols, n) % 13 - 6).astype(np.int8)
    qt_int = quant.QuantizedTensor(qi.reshape(-1), None, np.ones(n, np.float32), cols, n)
    got = quant.matmul_dequant_i8(ai, rows, cols, qt_int, ctx).reshape(rows, n)
    assert (got == ai.astype(np.int64) @ qi.astype(np.int64)).all()
    qt.free_gpu()
    qt_int.free_gpu()


@pytest.mark.parametrize("m,k,n", [
    (2, 2176, 4112), (16, 4224, 8208), (16, 2176, 12304), (5, 1152, 12304), (16, 1024, 12304),   # one tile of rows
    (17, 1024, 4096), (32, 300, 700), (19, 128, 520), (17, 1153, 8192), (32, 2048, 8208), (20, 2176, 4112), (32, 2176, 12290),
    (33, 1024, 8208), (64, 1000, 8192), (40, 130, 700), (48, 2048, 4112), (64, 4200, 8208), (33, 1536, 4000),
])
def test_few_rows_launch_shapes_bit_exact(ctx, orc, m, k, n):
    """Both sides of every line of the few-row launch's rule (16-row weight tiles against CUs, units of K), with ragged
    rows, K and columns.  The integers are exact in f64 and the scales are applied in one order, so the bits are determined."""
    from peregrine_amd import quant
    say(f"few rows m={m} k={k} n={n}")
    rng = np.random.default_rng(m * 7 + k + n)
    qt = quant.quantize_weights(rng.uniform(-0.05, 0.05, (k, n)).astype(np.float32), k, n, ctx)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::53] *= 20.0
    q, s = orc.quantize_activations(a, m, k)
    acc = np.asarray(q, np.float64).reshape(m, k) @ np.asarray(qt.data_i8, np.float64).reshape(k, n)
    want = acc.astype(np.float32) * np.asarray(s, np.float32)[:, None] * np.asarray(qt.scales, np.float32)[None, :]
    got = np.asarray(quant.matmul_quantized(a, m, k, qt, ctx), np.float32).reshape(m, n)
    assert (bits(got) == bits(want)).all()


@pytest.mark.parametrize("m,k,n", [
    (2, 512, 16400), (16, 512, 32800), (5, 640, 16400), (3, 640, 65552), (16, 768, 24576), (9, 2100, 24592), (16, 640, 32784), (2, 640, 49168),
    (16, 4200, 16400), (7, 4224, 32784),                                                                              # one tile of rows
    (17, 500, 32768), (32, 130, 32784), (20, 640, 16400), (31, 640, 32784), (32, 700, 49168), (17, 2176, 81936),       # two
    (33, 512, 16400), (64, 640, 24576), (48, 640, 24592), (50, 640, 32784), (64, 700, 49168), (33, 640, 65552),        # four
    (40, 2176, 65552), (64, 2200, 73744), (35, 2176, 98320),
])
def test_few_rows_over_wide_weights_bit_exact(ctx, orc, m, k, n):
    """Both sides of the lines between the few-row launch's shapes beyond 16384 columns (workgroups of 32 columns a CU),
    ragged rows, K and columns; at columns of the first, middle and last tiles."""
    from peregrine_amd import quant
    say(f"few rows over wide weights m={m} k={k} n={n}")
    rng = np.random.default_rng(m * 7 + k + n)
    q = rng.integers(-127, 128, (k, n), dtype=np.int8)
    scales = rng.uniform(0.5e-3, 2e-3, n).astype(np.float32)
    qt = quant.QuantizedTensor(q.reshape(-1), None, scales, k, n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::53] *= 20.0
    got = np.asarray(quant.matmul_quantized(a, m, k, qt, ctx), np.float32).reshape(m, n)
    cols = np.unique(np.r_[0:70, n // 2 : n // 2 + 40, n - 300 : n, rng.integers(0, n, 400)])
    qa, s = orc.quantize_activations(a, m, k)
    acc = np.asarray(qa, np.float64).reshape(m, k) @ q[:, cols].astype(np.float64)
    want = acc.astype(np.float32) * np.asarray(s, np.float32)[:, None] * scales[cols][None, :]
    assert (bits(got[:, cols]) == bits(want)).all()
    assert (np.abs(got).max(axis=0) > 0).all(), "a column was left out"
    qt.free_gpu()


@pytest.mark.parametrize("m,k,n", [
    (2, 4, 1), (3, 5, 15), (4, 7, 17), (8, 127, 16), (5, 128, 33), (2, 129, 256),                # part vectors, part tiles
    (4, 515, 64), (4, 516, 64), (2, 1027, 100), (3, 1028, 100), (4, 2051, 40), (4, 2052, 40),    # vectors to a lane; past the rule
    (8, 515, 64), (6, 516, 64), (8, 1027, 100), (5, 1028, 100), (8, 1539, 40), (7, 1540, 40),
    (4, 1027, 16383), (4, 1027, 16384), (4, 1028, 8191), (4, 1028, 8192),                         # columns, both sides
    (5, 771, 8191), (5, 771, 8192), (8, 772, 4095), (8, 772, 4096),
])
def test_short_f32_rows_bit_exact(ctx, orc, m, k, n):
    """Rows that every workgroup quantises for itself, at the edges of a lane's vectors and of the rule, alone and as
    two weights over one input, on device pointers; with a row of zeros, a NaN and halves that round away from zero."""
    from devbuf import DevBuf
    from peregrine_amd import quant, _ffi
    say(f"short f32 rows m={m} k={k} n={n}")
    rng = np.random.default_rng(m + 10 * k + n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::53] *= 20.0
    a[1] = 0.0
    a[0, :3] = 127.0, 63.5, np.nan
    a[0] = np.clip(a[0], -127, 127)
    a_dev = DevBuf(ctx, host=a)
    qa, s = orc.quantize_activations(a, m, k)
    cols = [n, max(1, n // 3)] if n < 4096 else [n - 16, 16]
    qts, wants = [], []
    for c in cols:
        q = rng.integers(-127, 128, (k, c), dtype=np.int8)
        scales = rng.uniform(0.5e-3, 2e-3, c).astype(np.float32)
        qts.append(quant.QuantizedTensor(q.reshape(-1), None, scales, k, c).to_gpu(ctx))
        acc = np.asarray(qa, np.float64).reshape(m, k) @ q.astype(np.float64)
        wants.append(acc.astype(np.float32) * np.asarray(s, np.float32)[:, None] * scales[None, :])
    outs = [DevBuf(ctx, nbytes=4 * m * c) for c in cols]
    for qt, want, out, c in zip(qts, wants, outs, cols):
        _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, a_dev.ptr, m, k, qt._gpu, out.ptr, None))
        assert (bits(out.to_host(np.float32).reshape(m, c)) == bits(want)).all()
    outs = [DevBuf(ctx, nbytes=4 * m * c) for c in cols]
    tab = lambda v: (C.c_void_p * len(v))(*v)
    _ffi.check(_ffi.lib.pg_matmul_quantized_multi_dev(ctx.handle, a_dev.ptr, m, k, tab([t._gpu.value for t in qts]), 2, tab([o.ptr.value for o in outs])))
    for want, out, c in zip(wants, outs, cols):
        assert (bits(out.to_host(np.float32).reshape(m, c)) == bits(want)).all()


@pytest.mark.parametrize("m,k,ns", [
    (33, 100, [17]), (33, 1000, [64, 33, 33]), (47, 4096, [300]), (48, 640, [515]), (49, 640, [515]), (64, 4096, [256, 64, 64]),
    (65, 384, [1030]), (96, 9300, [48]), (97, 2050, [700, 700]), (128, 1024, [1024]), (129, 511, [2000, 499, 499]), (144, 4096, [129]),
    (250, 1500, [333]), (256, 4097, [200, 50, 50]), (257, 260, [40]), (385, 2048, [250]), (511, 4096, [96]), (512, 1000, [130, 130]),
    (513, 1000, [130, 130]), (300, 300, [5000, 1250, 1250]), (40, 9216, [100]), (60, 256, [9000, 9000]),      # other routes beside them
])
def test_groups_of_rows_bit_exact(ctx, orc, m, k, ns):
    """33 to 512 rows in groups of 32, 48 and 64 over one to three weights, whole and part groups, one launch and the tiles beside
    it; the accumulators too where there is one weight."""
    from devbuf import DevBuf
    from peregrine_amd import quant, _ffi
    say(f"groups of rows m={m} k={k} ns={ns}")
    rng = np.random.default_rng(m + 10 * k + ns[0])
    a = rng.standard_normal((m, k)).astype(np.float32)
    a[:, ::53] *= 20.0
    a[m // 2] = 0.0
    a_dev = DevBuf(ctx, host=a)
    qa, s = orc.quantize_activations(a, m, k)
    qts, wants, accs = [], [], []
    for c in ns:
        q = rng.integers(-127, 128, (k, c), dtype=np.int8)
        scales = rng.uniform(0.5e-3, 2e-3, c).astype(np.float32)
        qts.append(quant.QuantizedTensor(q.reshape(-1), None, scales, k, c).to_gpu(ctx))
        acc = np.asarray(qa, np.float64).reshape(m, k) @ q.astype(np.float64)
        accs.append(acc)
        wants.append(acc.astype(np.float32) * np.asarray(s, np.float32)[:, None] * scales[None, :])
    outs = [DevBuf(ctx, nbytes=4 * m * c) for c in ns]
    tab = lambda v: (C.c_void_p * len(v))(*v)
    _ffi.check(_ffi.lib.pg_matmul_quantized_multi_dev(ctx.handle, a_dev.ptr, m, k, tab([t._gpu.value for t in qts]), len(ns), tab([o.ptr.value for o in outs])))
    for want, out, c in zip(wants, outs, ns):
        assert (bits(out.to_host(np.float32).reshape(m, c)) == bits(want)).all()
    acc_dev = DevBuf(ctx, nbytes=4 * m * ns[0])
    _ffi.check(_ffi.lib.pg_matmul_quantized_dev(ctx.handle, a_dev.ptr, m, k, qts[0]._gpu, outs[0].ptr, acc_dev.ptr))
    assert (bits(outs[0].to_host(np.float32).reshape(m, ns[0])) == bits(wants[0])).all()
    assert (acc_dev.to_host(np.int32).reshape(m, ns[0]) == accs[0].astype(np.int32)).all()


@pytest.mark.parametrize("m,k", [(1, 768), (1, 4096), (2, 128), (3, 768), (4, 2048), (5, 768), (8, 1536), (8, 640), (17, 512), (40, 1024), (1, 20000)])
@pytest.mark.parametrize("shift", [0, 1, -1])
def test_w8a8_over_its_own_rows_bit_exact(ctx, orc, m, k, shift):
    """A result over the rows it is made from, whole or one row further on: no workgroup may store before every other has read
    the rows.  A weight alone, in the fixed scratch, and the first and the last of two over one input."""
    from devbuf import DevBuf
    from peregrine_amd import quant, _ffi
    say(f"W8A8 over its own rows m={m} k={k} shift={shift}")
    rng = np.random.default_rng(m + 10 * k)
    n = k if k < 20000 else 3000
    a = rng.standard_normal((m, k)).astype(np.float32)
    q = rng.integers(-127, 128, (k, n), dtype=np.int8)
    scales = rng.uniform(0.5e-3, 2e-3, n).astype(np.float32)
    qt = quant.QuantizedTensor(q.reshape(-1), None, scales, k, n).to_gpu(ctx)
    other = quant.QuantizedTensor(np.ascontiguousarray(q[:, ::-1]).reshape(-1), None, scales, k, n).to_gpu(ctx)
    qa, s = orc.quantize_activations(a, m, k)
    acc = np.asarray(qa, np.float64).reshape(m, k) @ q.astype(np.float64)
    want = acc.astype(np.float32) * np.asarray(s, np.float32)[:, None] * scales[None, :]
    wants = want, acc[:, ::-1].astype(np.float32) * np.asarray(s, np.float32)[:, None] * scales[None, :]
    L = _ffi.lib
    tab = lambda v: (C.c_void_p * len(v))(*v)

    def check(call, w):
        buf = DevBuf(ctx, host=np.concatenate([np.zeros(k, np.float32), a.reshape(-1), np.zeros(k, np.float32)]))
        aside = DevBuf(ctx, nbytes=4 * m * n)
        rows = buf.ptr.value + 4 * k
        _ffi.check(call(C.c_void_p(rows), rows + 4 * k * shift, aside.ptr.value))
        got = buf.to_host(np.float32)[k + k * shift:][: m * n].reshape(m, n)
        assert (bits(got) == bits(wants[w])).all()
        return aside.to_host(np.float32).reshape(m, n)

    check(lambda x, out, _: L.pg_matmul_quantized_dev(ctx.handle, x, m, k, qt._gpu, C.c_void_p(out), None), 0)
    check(lambda x, out, _: L.pg_matmul_quantized_fixed_scratch_dev(ctx.handle, x, m, k, qt._gpu, C.c_void_p(out)), 0)
    both = tab([qt._gpu.value, other._gpu.value])
    aside = check(lambda x, out, at: L.pg_matmul_quantized_multi_dev(ctx.handle, x, m, k, both, 2, tab([out, at])), 0)
    assert (bits(aside) == bits(wants[1])).all()
    aside = check(lambda x, out, at: L.pg_matmul_quantized_multi_dev(ctx.handle, x, m, k, both, 2, tab([at, out])), 1)
    assert (bits(aside) == bits(wants[0])).all()


@pytest.mark.parametrize("m,k,ns,apart", [(46, 13300, [294, 9512], 0), (135, 10836, [628, 8185], 0), (63, 13958, [8390, 421, 363], 0), (65, 10836, [628, 8185], 0)])
def test_several_weights_some_split_over_k_bit_exact(ctx, orc, m, k, ns, apart):
    """Weights over one long K, some of few columns: one launch for all of them, none apart and split over K; and the bits."""
    from peregrine_amd import quant, _ffi
    say(f"several weights, split over K m={m} k={k} ns={ns}")
    rng = np.random.default_rng(m + 10 * k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    a_dev = DevBuf(ctx, host=a)
    qa, s = orc.quantize_activations(a, m, k)
    qts, wants = [], []
    for c in ns:
        q = rng.integers(-127, 128, (k, c), dtype=np.int8)
        scales = rng.uniform(0.5e-3, 2e-3, c).astype(np.float32)
        qts.append(quant.QuantizedTensor(q.reshape(-1), None, scales, k, c).to_gpu(ctx))
        acc = np.asarray(qa, np.float64).reshape(m, k) @ q.astype(np.float64)
        wants.append(acc.astype(np.float32) * np.asarray(s, np.float32)[:, None] * scales[None, :])
    outs = [DevBuf(ctx, nbytes=4 * m * c) for c in ns]
    tab = lambda v: (C.c_void_p * len(v))(*v)
    ctx.profile_begin()
    _ffi.check(_ffi.lib.pg_matmul_quantized_multi_dev(ctx.handle, a_dev.ptr, m, k, tab([t._gpu.value for t in qts]), len(ns), tab([o.ptr.value for o in outs])))
    assert ctx.profile_end().get("gemm_w8a8_finish", (0, 0))[1] == apart
    for want, out, c in zip(wants, outs, ns):
        assert (bits(out.to_host(np.float32).reshape(m, c)) == bits(want)).all()
