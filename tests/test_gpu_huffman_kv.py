"""GPU parity of the Huffman-coded KV cache against the CPU oracle, through the C ABI.
Bar: bit-exact everywhere (scales, code table, bitstream bytes, decoded f32 values, the
cache's lengths and what get_kv returns)."""
import ctypes as C
import sys

import numpy as np
import pytest

from devbuf import DevBuf
from test_oracle_formats_pins import parity_random_data

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _same_chunk(chunk, want):
    bits, scales, codebook = want[:3]
    assert chunk.codebook == codebook.tobytes()
    assert (chunk.scales.view(np.uint32) == scales.view(np.uint32)).all()
    assert chunk.bitstream == bits


def _chunk_data(kind, t, h, d, seed):
    rng = np.random.default_rng(seed)
    n = t * h * d
    if kind == "normal":
        return rng.standard_normal(n).astype(np.float32)
    if kind == "uniform":
        return parity_random_data(n, seed)
    if kind == "scaled_heads":                     # heads of very different magnitude, one of them all zero
        x = rng.standard_normal((h, t * d)).astype(np.float32) * (10.0 ** rng.integers(-6, 6, (h, 1))).astype(np.float32)
        x[rng.integers(0, h)] = 0.0
        return x.reshape(-1)
    if kind == "constant":
        return np.full(n, -0.75, np.float32)
    if kind == "special":                          # NaN is skipped by the maximum and becomes 0; halves round away from zero
        x = rng.standard_normal(n).astype(np.float32)
        x[::7] = np.nan
        x[1::11] = 0.0
        if n > 4:
            x[2], x[3] = 127.0, 63.5
        return x
    raise AssertionError(kind)


@pytest.mark.parametrize("kind,t,h,d", [
    ("uniform", 32, 4, 16),          # tests/huffman_parity.rs:133-158
    ("normal", 5, 3, 7), ("normal", 1, 1, 1), ("normal", 16, 2, 8), ("normal", 256, 2, 8),
    ("normal", 31, 3, 43),           # 3999 symbols: one encoder workgroup with a ragged tail
    ("normal", 64, 2, 128),          # a table whose reference form over-subscribes the code: repaired
    ("normal", 256, 8, 128),         # 262144 symbols, 64 encoder workgroups
    ("scaled_heads", 40, 6, 64), ("constant", 7, 5, 3), ("special", 9, 2, 16), ("special", 300, 3, 64),
])
def test_compress_chunk_is_the_oracle_s(ctx, orc, kind, t, h, d):
    from peregrine_amd import huffman
    say(f"huffman kv compress_chunk {kind} tokens={t} heads={h} head_dim={d}")
    data = _chunk_data(kind, t, h, d, 1000 + t + h + d)
    want = orc.huffman_kv_compress_chunk(data, t, h, d)
    chunk = huffman.HuffmanKVCache.compress_chunk(data, t, h, d, ctx)
    assert (chunk.num_tokens, chunk.num_heads, chunk.head_dim) == (t, h, d)
    _same_chunk(chunk, want)
    got = huffman.HuffmanKVCache.decompress_chunk(chunk)
    ref = orc.huffman_kv_decompress_chunk(*want[:3], t, h, d)
    assert (got.view(np.uint32) == ref.view(np.uint32)).all()
    # a chunk rebuilt from the oracle's parts decodes to the same values
    again = huffman.CompressedChunk.from_parts(want[0], want[1], want[2], t, h, d, ctx)
    assert (huffman.HuffmanKVCache.decompress_chunk(again).view(np.uint32) == ref.view(np.uint32)).all()
    if kind in ("uniform", "normal"):              # the reference's bound, and the half step that rounding to nearest gives
        err = np.abs(got - data).reshape(h, -1).max(axis=1)
        assert (err <= want[1] + 1e-5).all() and (err <= want[1] * 0.5 * (1 + 1e-6)).all()


def test_reference_unit_test_chunk(ctx, orc):
    """src/huffman.rs:879-905."""
    from peregrine_amd import huffman
    h, d, t = 2, 8, 16
    data = np.array([((i * 13 + 7) % 100) / 50.0 - 1.0 for i in range(h * t * d)], np.float32)
    chunk = huffman.HuffmanKVCache.compress_chunk(data, t, h, d, ctx)
    _same_chunk(chunk, orc.huffman_kv_compress_chunk(data, t, h, d))
    rec = huffman.HuffmanKVCache.decompress_chunk(chunk)
    absmax = np.abs(data).reshape(h, -1).max(axis=1)
    assert (np.abs(rec - data).reshape(h, -1).max(axis=1) <= absmax / 127 + 1e-5).all()


def test_empty_chunks_and_errors(ctx, orc):
    from peregrine_amd import huffman, _ffi
    for t, h, d in ((0, 2, 4), (3, 0, 4), (3, 2, 0)):
        chunk = huffman.HuffmanKVCache.compress_chunk(np.zeros(0, np.float32), t, h, d, ctx)
        want = orc.huffman_kv_compress_chunk(np.zeros(0, np.float32), t, h, d)
        _same_chunk(chunk, want)
        assert chunk.bitstream == b"" and huffman.HuffmanKVCache.decompress_chunk(chunk).size == 0
    with pytest.raises(ValueError):
        huffman.HuffmanKVCache.compress_chunk(np.zeros(5, np.float32), 1, 2, 3, ctx)      # assert_eq!(data.len(), total)
    with pytest.raises(_ffi.PeregrineError):
        huffman.HuffmanKVCache(2, 4, 8, 0, ctx)                                           # the reference's append would never return
    # a stream that is too short for its symbol count, and a codebook that cannot produce it
    bits, scales, codebook, _ = orc.huffman_kv_compress_chunk(np.linspace(-1, 1, 64, dtype=np.float32), 8, 2, 4)
    short = huffman.CompressedChunk.from_parts(bits[:len(bits) // 2], scales, codebook, 8, 2, 4, ctx)
    with pytest.raises(_ffi.PeregrineError):
        huffman.HuffmanKVCache.decompress_chunk(short)
    one = np.zeros(256, np.uint8)
    one[128] = 1
    wrong = huffman.CompressedChunk.from_parts(bytes([0xFF] * 8), scales, one, 8, 2, 4, ctx)
    with pytest.raises(_ffi.PeregrineError):
        huffman.HuffmanKVCache.decompress_chunk(wrong)


def test_chunks_from_and_to_strided_device_memory(ctx, orc):
    """The `_dev` entry points: heads `head_stride` floats apart on both sides, as in a StandardKVCache."""
    from peregrine_amd import huffman, _ffi
    t, h, d, stride = 24, 3, 32, 24 * 32 + 160
    rng = np.random.default_rng(8)
    padded = rng.standard_normal((h, stride)).astype(np.float32)
    data = padded[:, :t * d].copy()
    src = DevBuf(ctx, host=padded)
    handle = C.c_void_p()
    _ffi.check(_ffi.lib.pg_huffman_kv_compress_chunk_dev(ctx.handle, src.ptr, stride, t, h, d, C.byref(handle)))
    chunk = huffman.CompressedChunk(handle, ctx)
    want = orc.huffman_kv_compress_chunk(data, t, h, d)
    _same_chunk(chunk, want)
    dst = DevBuf(ctx, host=np.full((h, stride), 7.0, np.float32))
    _ffi.check(_ffi.lib.pg_huffman_kv_decompress_chunk_dev(ctx.handle, chunk._h, dst.ptr, stride))
    ctx.sync()
    got = dst.to_host(np.float32).reshape(h, stride)
    ref = orc.huffman_kv_decompress_chunk(*want[:3], t, h, d).reshape(h, t * d)
    assert (got[:, :t * d].view(np.uint32) == ref.view(np.uint32)).all() and (got[:, t * d:] == 7.0).all()
    with pytest.raises(_ffi.PeregrineError):
        _ffi.check(_ffi.lib.pg_huffman_kv_decompress_chunk_dev(ctx.handle, chunk._h, dst.ptr, t * d - 1))


def test_reference_cache_tests(ctx, orc):
    from peregrine_amd import huffman
    # src/huffman.rs:850-876
    c = huffman.HuffmanKVCache(2, 4, 8, 4, ctx)
    c.append(np.full(32, 1.0, np.float32), np.full(32, 2.0, np.float32), 4)
    assert (c.len(), c.compressed_len) == (4, 0)
    c.append(np.full(32, 3.0, np.float32), np.full(32, 4.0, np.float32), 4)
    assert (c.len(), c.compressed_len) == (8, 4)
    k, v = c.get_kv()
    assert k.size == v.size == 2 * 8 * 4
    assert (k.reshape(2, 8, 4)[:, :4] == 1.0).all() and (k.reshape(2, 8, 4)[:, 4:] == 3.0).all()
    assert (v.reshape(2, 8, 4)[:, :4] == 2.0).all() and (v.reshape(2, 8, 4)[:, 4:] == 4.0).all()
    # tests/huffman_parity.rs:160-186
    c = huffman.HuffmanKVCache(2, 8, 16, 8, ctx)
    o = orc.HuffmanKVCache(2, 8, 16, 8)
    for batch in range(4):
        k, v = parity_random_data(2 * 8 * 8, 100 + batch), parity_random_data(2 * 8 * 8, 200 + batch)
        c.append(k, v, 8)
        o.append(k, v, 8)
    assert c.len() == 32 and c.compressed_len > 0 and c.compressed_len == o.compressed_len
    for got, want in zip(c.get_kv(), o.get_kv()):
        assert got.size == 2 * 32 * 8 and (got.view(np.uint32) == want.view(np.uint32)).all()
    assert huffman.HuffmanKVCache(1, 1, 3, 10, ctx).compress_threshold == 10             # src/huffman.rs:535


@pytest.mark.parametrize("heads,hd,thr,chunk,appends", [
    (2, 8, 16, 8, (8, 8, 8, 8)),
    (3, 4, 10, 4, (1, 7, 2, 30, 5, 1, 0, 3)),      # one append that cuts several chunks, an empty append
    (1, 16, 0, 5, (3, 3, 3, 20)),                  # threshold below the chunk size: raised to it
    (2, 2, 6, 6, (13,)),
    (2, 8, 64, 4, (70, 3, 3, 1)),                  # a window much longer than a chunk: it moves to the front in many slices
    (8, 128, 512, 256, (300, 1, 1, 400, 1)),       # a Llama-sized cache: 262144 symbols per chunk
    (2, 16, 8, 4, (5,) * 60),                      # 74 chunks per side: get_kv decodes 148 streams, each under its own table, in one pass
])
def test_cache_follows_the_oracle(ctx, orc, heads, hd, thr, chunk, appends):
    from peregrine_amd import huffman
    say(f"huffman kv cache heads={heads} head_dim={hd} threshold={thr} chunk={chunk} appends={appends}")
    rng = np.random.default_rng(heads * 1000 + hd)
    c, o = huffman.HuffmanKVCache(heads, hd, thr, chunk, ctx), orc.HuffmanKVCache(heads, hd, thr, chunk)
    assert c.compress_threshold == o.compress_threshold
    for n in appends:
        k = rng.standard_normal((heads, n, hd)).astype(np.float32)
        v = (rng.standard_normal((heads, n, hd)) * 3).astype(np.float32)
        c.append(k, v, n)
        o.append(k, v, n)
        assert (c.len(), c.compressed_len, c.hot_len, len(c.k_chunks)) == (o.len, o.compressed_len, o.hot_len, o.num_chunks)
        for got, want in zip(c.get_kv(), o.get_kv()):
            assert (got.view(np.uint32) == want.view(np.uint32)).all()
    for side, chunks in ((0, c.k_chunks), (1, c.v_chunks)):
        for i, ch in enumerate(chunks):
            bits, scales, codebook, tokens = o.chunk(side, i)
            assert ch.num_tokens == tokens
            _same_chunk(ch, (bits, scales, codebook))


def test_cache_on_device_pointers(ctx, orc):
    """append_dev / get_kv_dev: the caller's tensors never leave the device."""
    from peregrine_amd import huffman, _ffi
    heads, hd = 4, 64
    c, o = huffman.HuffmanKVCache(heads, hd, 48, 32, ctx), orc.HuffmanKVCache(heads, hd, 48, 32)
    rng = np.random.default_rng(21)
    for n in (40, 1, 1, 70, 1):
        k, v = rng.standard_normal((heads, n, hd)).astype(np.float32), rng.standard_normal((heads, n, hd)).astype(np.float32)
        dk, dv = DevBuf(ctx, host=k), DevBuf(ctx, host=v)
        _ffi.check(_ffi.lib.pg_huffman_kv_cache_append_dev(ctx.handle, c._h, dk.ptr, dv.ptr, n))
        o.append(k, v, n)
    assert (c.len(), c.compressed_len) == (o.len, o.compressed_len)
    n = heads * c.len() * hd
    out_k, out_v = DevBuf(ctx, nbytes=4 * n), DevBuf(ctx, nbytes=4 * n)
    _ffi.check(_ffi.lib.pg_huffman_kv_cache_get_kv_dev(ctx.handle, c._h, out_k.ptr, out_v.ptr))
    ctx.sync()
    want_k, want_v = o.get_kv()
    assert (out_k.to_host(np.float32).view(np.uint32) == want_k.view(np.uint32)).all()
    assert (out_v.to_host(np.float32).view(np.uint32) == want_v.view(np.uint32)).all()


@pytest.mark.parametrize("heads,hd,chunk,chunks", [
    (1, 1, 4095, 2), (1, 1, 4096, 2), (1, 1, 4097, 2),     # a histogram run of 4096 values, one less, one more
    (1, 4, 4096, 1), (1, 4, 4097, 1), (3, 1, 5462, 1),     # a decoder workgroup of 16384, and 2 (with a head cut by the runs) past it
    (1, 64, 1, 45), (5, 3, 2, 40),                         # more chunks in one batch than one encoder launch places
    (1, 1, 262144, 1), (1, 1, 262145, 1),                  # 64 histograms, which the table kernel keeps, and one more
    (1, 1, 65536, 1), (1, 1, 65537, 1),                    # the longest head whose maximum every workgroup finds, and one more
    (3, 1, 2047, 2), (3, 1, 2048, 2),                      # heads by a wavefront, and by the workgroup
    (1, 1, 4096, 256), (1, 1, 4096, 257),                  # as many workgroups as take that route, and more
    (2, 2, 70000, 1),                                      # 69 runs of a head's values, several rounds of the maximum
])
@pytest.mark.parametrize("kind", ["normal", "steep", "two"])
def test_batches_and_run_edges(ctx, orc, heads, hd, chunk, chunks, kind):
    """One append that cuts `chunks` whole chunks at the edges of the batch's runs, workgroups and launches; `steep` has
    frequencies that halve from value to value (codes past the limit of 12 bits, repaired), `two` has two values."""
    from peregrine_amd import huffman
    say(f"huffman kv batch heads={heads} head_dim={hd} chunk={chunk} x {chunks} {kind}")
    rng = np.random.default_rng(chunk + heads)
    n = chunk * chunks
    if kind == "normal":
        k, v = (rng.standard_normal((heads, n, hd)).astype(np.float32) for _ in range(2))
    elif kind == "steep":
        k, v = (np.minimum(rng.geometric(0.5, (heads, n, hd)), 40).astype(np.float32) for _ in range(2))
        k[:, 0], v[:, 0] = 40.0, 40.0
    else:
        k, v = (rng.integers(0, 2, (heads, n, hd)).astype(np.float32) for _ in range(2))
    c, o = huffman.HuffmanKVCache(heads, hd, chunk, chunk, ctx), orc.HuffmanKVCache(heads, hd, chunk, chunk)
    c.append(k, v, n)
    o.append(k, v, n)
    assert (c.len(), c.compressed_len, len(c.k_chunks)) == (o.len, o.compressed_len, chunks)
    for got, want in zip(c.get_kv(), o.get_kv()):
        assert (got.view(np.uint32) == want.view(np.uint32)).all()
    for side, made in ((0, c.k_chunks), (1, c.v_chunks)):
        for i in {0, chunks // 2, chunks - 1}:
            _same_chunk(made[i], o.chunk(side, i)[:3])


def _counts(kind):
    """How often each of the values -127 .. 127 occurs (127 always does: the scale is then 1 and a value its own code)."""
    i = np.arange(255, dtype=np.int64)
    if kind == "equal":                                    # every tree ties: more pairs in a round than a wavefront takes
        return np.full(255, 9)
    if kind == "ties":                                     # leaves and nodes of one weight, leaf first
        return 1 << (i // 20)
    if kind == "fibonacci":                                # one pair a round, the deepest tree
        c = np.zeros(255, np.int64)
        c[-26:] = [1, 1] + [0] * 24
        for j in range(255 - 24, 255):
            c[j] = c[j - 1] + c[j - 2]
        return c
    if kind == "ramp":
        return i % 83 + 1
    c = np.zeros(255, np.int64)
    c[254] = 5                                             # one symbol
    return c


@pytest.mark.parametrize("kind", ["equal", "ties", "fibonacci", "ramp", "one"])
@pytest.mark.parametrize("total", [0, (1 << 23) - 1, 1 << 23])
def test_tables_at_the_edges_of_the_merges(ctx, orc, kind, total):
    """Histograms that the merge rounds can go wrong at, as they are and brought to the total at which their keys
    become 64 bits wide, and to one value less."""
    from peregrine_amd import huffman
    say(f"huffman kv table {kind} total={total}")
    counts = _counts(kind)
    if total:
        counts = counts * (total // counts.sum())
        counts[254] += total - counts.sum()
    data = np.repeat(np.arange(-127, 128), counts).astype(np.float32)
    chunk = huffman.HuffmanKVCache.compress_chunk(data, len(data), 1, 1, ctx)
    _same_chunk(chunk, orc.huffman_kv_compress_chunk(data, len(data), 1, 1))
    assert (huffman.HuffmanKVCache.decompress_chunk(chunk) == data).all()


@pytest.mark.parametrize("heads,hd,thr,chunk,appends,skew", [
    (4, 64, 48, 32, (40, 1, 1, 70, 1, 0, 200), 0),   # chunks of old rows, of old and new ones, of new ones alone
    (4, 64, 48, 32, (40, 1, 70), 1),                 # rows that start off a 16-byte boundary
    (3, 7, 5, 5, (3, 1, 1, 1, 24, 2), 0),            # no four values of one head
    (2, 6, 4, 2, (1, 1, 1, 1, 3, 8), 0),             # whole quadruples in a chunk, not in the window's rows
    (1, 1, 1, 1, (1100, 3), 0),                      # more chunks than one batch takes
    (8, 128, 512, 256, (500, 500, 1100), 0),
    (1, 2, 40000, 40000, (30000, 20000, 1), 0),      # heads that a launch of their own finds the maximum of
    (1, 1, 70001, 70001, (30001, 50000), 0),
])
def test_device_rows_are_written_with_the_maximum(ctx, orc, heads, hd, thr, chunk, appends, skew):
    """append_dev where it cuts chunks: the launch that finds the chunks' maxima also writes the new rows."""
    from peregrine_amd import huffman, _ffi
    say(f"huffman kv device rows heads={heads} head_dim={hd} threshold={thr} chunk={chunk} appends={appends} skew={skew}")
    c, o = huffman.HuffmanKVCache(heads, hd, thr, chunk, ctx), orc.HuffmanKVCache(heads, hd, thr, chunk)
    rng = np.random.default_rng(hd)
    for n in appends:
        k, v = (rng.standard_normal(skew + heads * n * hd + 1).astype(np.float32) for _ in range(2))
        dk, dv = DevBuf(ctx, host=k), DevBuf(ctx, host=v)
        at = [C.c_void_p(d.ptr.value + 4 * skew) for d in (dk, dv)]
        _ffi.check(_ffi.lib.pg_huffman_kv_cache_append_dev(ctx.handle, c._h, *at, n))
        o.append(*(x[skew:skew + heads * n * hd].reshape(heads, n, hd) for x in (k, v)), n)
        assert (c.len(), c.compressed_len) == (o.len, o.compressed_len)
        for got, want in zip(c.get_kv(), o.get_kv()):
            assert (got.view(np.uint32) == want.view(np.uint32)).all()


@pytest.mark.parametrize("heads,hd,thr,chunk", [(2, 16, 24, 16), (3, 7, 5, 5), (4, 64, 96, 64)])
def test_streams_longer_than_the_last(ctx, orc, heads, hd, thr, chunk):
    """Batches whose streams take more than the one before led to expect are coded twice, the window moved once; up to
    two batches of more chunks than one encoder launch places."""
    from peregrine_amd import huffman
    say(f"huffman kv lengthening streams heads={heads} head_dim={hd} threshold={thr} chunk={chunk}")
    rng = np.random.default_rng(heads)
    c, o = huffman.HuffmanKVCache(heads, hd, thr, chunk, ctx), orc.HuffmanKVCache(heads, hd, thr, chunk)
    for kind, n in (("two", 3 * chunk), ("two", chunk + 1), ("normal", 2 * chunk), ("two", chunk), ("normal", chunk - 1), ("few", 40 * chunk), ("normal", 41 * chunk)):
        if kind == "normal":
            k, v = (rng.standard_normal((heads, n, hd)).astype(np.float32) for _ in range(2))
        else:
            k, v = (rng.integers(0, 2 if kind == "two" else 9, (heads, n, hd)).astype(np.float32) for _ in range(2))
        c.append(k, v, n)
        o.append(k, v, n)
        assert (c.len(), c.compressed_len, c.hot_len) == (o.len, o.compressed_len, o.hot_len)
        for got, want in zip(c.get_kv(), o.get_kv()):
            assert (got.view(np.uint32) == want.view(np.uint32)).all()
    for side, chunks in ((0, c.k_chunks), (1, c.v_chunks)):
        for i, ch in enumerate(chunks):
            _same_chunk(ch, o.chunk(side, i)[:3])


@pytest.mark.parametrize("heads,hd,thr,chunk", [(2, 16, 24, 16), (4, 64, 96, 64), (8, 128, 512, 256)])
def test_sides_of_different_streams(ctx, orc, heads, hd, thr, chunk):
    """Keys and values that code to very different lengths, alike from append to append, in turn the one and the other, and in
    batches of which one chunk alone outgrows its room: what the device makes of its sizes is what the host does."""
    from peregrine_amd import huffman
    say(f"huffman kv sides heads={heads} head_dim={hd} threshold={thr} chunk={chunk}")
    rng = np.random.default_rng(heads + 7)
    c, o = huffman.HuffmanKVCache(heads, hd, thr, chunk, ctx), orc.HuffmanKVCache(heads, hd, thr, chunk)
    few = lambda n: rng.integers(0, 2, (heads, n, hd)).astype(np.float32)
    many = lambda n: rng.standard_normal((heads, n, hd)).astype(np.float32)
    late = lambda n: np.concatenate([few(n - n // 3), many(n // 3)], 1)
    for k, v, n in ((few, many, thr), (few, many, chunk), (few, many, chunk + 3), (many, few, chunk), (many, few, 2 * chunk), (many, late, 3 * chunk),
                    (late, many, 3 * chunk), (few, few, chunk), (few, few, chunk), (many, many, 35 * chunk), (many, many, 35 * chunk)):
        k, v = k(n), v(n)
        c.append(k, v, n)
        o.append(k, v, n)
        assert (c.len(), c.compressed_len, c.hot_len) == (o.len, o.compressed_len, o.hot_len)
        for got, want in zip(c.get_kv(), o.get_kv()):
            assert (got.view(np.uint32) == want.view(np.uint32)).all()
    for side, chunks in ((0, c.k_chunks), (1, c.v_chunks)):
        for i in {0, len(chunks) // 2, len(chunks) - 1}:
            _same_chunk(chunks[i], o.chunk(side, i)[:3])


@pytest.mark.parametrize("heads,hd,thr,chunk", [
    (2, 8, 36, 4),     # chains of 9 steps of 16 bytes: two rounds of 4 loads and one more
    (3, 7, 40, 8),     # rows that 16 bytes do not divide, the last chains shorter
    (1, 1, 33, 1),     # one value a chain step
    (2, 64, 520, 512), # a move shorter than its distance
    (8, 128, 300, 256),
])
def test_the_window_moves_and_grows_in_one_launch(ctx, orc, heads, hd, thr, chunk):
    """What stays in the window is the same bits after each move to the front, whatever the number of steps, and after each growth."""
    from peregrine_amd import huffman
    say(f"huffman kv window heads={heads} head_dim={hd} threshold={thr} chunk={chunk}")
    rng = np.random.default_rng(thr)
    c, o = huffman.HuffmanKVCache(heads, hd, thr, chunk, ctx), orc.HuffmanKVCache(heads, hd, thr, chunk)
    for n in (3, thr - 4, 1, chunk, chunk // 2 + 1, 2 * chunk + 1, 1, 2 * thr):
        k, v = (rng.standard_normal((heads, n, hd)).astype(np.float32) for _ in range(2))
        c.append(k, v, n)
        o.append(k, v, n)
        assert (c.len(), c.compressed_len, c.hot_len) == (o.len, o.compressed_len, o.hot_len)
        for got, want in zip(c.get_kv(), o.get_kv()):
            assert (got.view(np.uint32) == want.view(np.uint32)).all()
