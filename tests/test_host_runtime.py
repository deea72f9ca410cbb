"""What the library does around its launches, followed without a GPU: the library's own objects, linked with a HIP runtime
on host memory that notes kernels instead of running them (tests/cpp/host_runtime.cpp).  Nothing here looks at a computed
number."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import helpers as H

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
LIB = os.path.join(CPP, "_build", "libperegrine_host.so")


NO_LIMIT = C.c_size_t(-1).value


class Host:
    """The library on the host runtime, one context to begin with."""

    def __init__(self):
        from peregrine_amd import _ffi
        if not os.path.exists(LIB):
            subprocess.check_call(["make", "-C", CPP])
        self.lib = C.CDLL(LIB)
        for name, args in _ffi.SIGNATURES.items():
            fn = getattr(self.lib, name)
            fn.argtypes, fn.restype = args, _ffi._OTHER_RESTYPE.get(name, C.c_int)
        for name in ("pghost_used", "pghost_frees", "pghost_bad_frees", "pghost_recorded", "pghost_copied", "pghost_num_launches"):
            getattr(self.lib, name).restype = C.c_size_t
        self.lib.pghost_limit.argtypes = [C.c_size_t]
        self.lib.pghost_fail_after.argtypes = self.lib.pghost_stream_bytes.argtypes = [C.c_size_t, C.c_size_t]
        self.lib.pghost_fail_after.restype = self.lib.pghost_stream_bytes.restype = None
        self.lib.pghost_limit.restype = self.lib.pghost_clear_launches.restype = self.lib.pghost_begin_capture.restype = None
        self.lib.pghost_begin_capture.argtypes = self.lib.pghost_end_capture.argtypes = [C.c_void_p]
        self.lib.pghost_launch.argtypes, self.lib.pghost_launch.restype = [C.c_size_t, C.POINTER(C.c_uint)], C.c_char_p
        self.ctx = self.new("pg_ctx_create", 0, None)

    def ok(self, name, *args):
        st = getattr(self.lib, name)(*args)
        assert st == 0, (name, st, self.lib.pg_last_error())

    def new(self, name, *args):
        h = C.c_void_p()
        self.ok(name, *args, C.byref(h))
        return h

    def alloc(self, floats):
        return self.new("pg_dev_alloc", self.ctx, floats * 4)

    def stream(self, ctx=None):
        return self.lib.pg_ctx_stream(ctx or self.ctx)

    def launches(self):
        grid, out = (C.c_uint * 3)(), []
        for i in range(self.lib.pghost_num_launches()):
            name = self.lib.pghost_launch(i, grid)
            out.append((name.decode(), tuple(grid)))
        return out

    def captured(self, fn, *args):
        """fn's status on a capturing stream, what the capture recorded, and whether it is still whole."""
        self.lib.pghost_begin_capture(self.stream())
        st = getattr(self.lib, fn)(*args)
        recorded = self.lib.pghost_recorded()
        return st, recorded, bool(self.lib.pghost_end_capture(self.stream()))

    def cache(self, heads, hd, tokens, ctx=None):
        c = self.new("pg_kv_cache_create", ctx or self.ctx, heads, hd)
        if tokens:
            rows = self.alloc(heads * hd * tokens)
            self.ok("pg_kv_cache_append_dev", ctx or self.ctx, c, rows, rows, tokens)
        return c

    def gguf(self, n, k):
        return self.new("pg_gguf_upload", self.ctx, bytes(H.pack_q4_0(np.zeros(n * k, np.float32))), 2, n, k)


@pytest.fixture()
def host():
    h = Host()
    h.lib.pghost_limit(NO_LIMIT)
    h.lib.pghost_fail_after(NO_LIMIT, NO_LIMIT)
    h.lib.pghost_stream_bytes(1000, 1000)
    h.lib.pghost_clear_launches()
    yield h
    assert h.lib.pghost_bad_frees() == 0
    h.lib.pg_ctx_destroy(h.ctx)


def test_cache_growth_is_refused_by_a_capture_whatever_the_pool_holds(host):
    heads, hd = 2, 64
    c = host.cache(heads, hd, 32)
    host.lib.pg_kv_cache_free(host.ctx, host.cache(heads, hd, 64))     # two blocks of the grown size in the pool
    row = host.alloc(heads * hd)
    st, recorded, whole = host.captured("pg_kv_cache_append_dev", host.ctx, c, row, row, 1)
    assert st == 2 and b"captur" in host.lib.pg_last_error() and recorded == 0 and whole
    assert host.lib.pg_kv_cache_len(c) == 32 and host.lib.pg_kv_cache_capacity(c) == 32
    host.ok("pg_kv_cache_append_dev", host.ctx, c, row, row, 1)        # eagerly it grows
    assert host.lib.pg_kv_cache_capacity(c) == 64
    st, recorded, whole = host.captured("pg_kv_cache_append_dev", host.ctx, c, row, row, 1)
    assert st == 0 and recorded == 1 and whole                         # with room there, it is one launch
    host.lib.pg_kv_cache_free(host.ctx, c)


@pytest.mark.parametrize("seq", [1, 4, 40])
def test_block_step_that_grows_its_cache_is_refused_by_a_capture(host, seq):
    d, nqh, nkvh, hd, ffn = 256, 4, 2, 64, 512
    shapes = [(nqh * hd, d), (nkvh * hd, d), (nkvh * hd, d), (d, nqh * hd), (ffn, d), (ffn, d), (d, ffn)]
    ws = [host.gguf(n, k) for n, k in shapes]
    b = host.new("pg_llama_block_create", host.ctx, d, nqh, nkvh, hd, ffn, 512, 10000.0, 1e-5)
    norm = np.ones(d, np.float32)
    host.ok("pg_llama_block_set_weights", host.ctx, b, *ws, norm.ctypes.data, norm.ctypes.data)
    x, out = host.alloc(64 * d), host.alloc(64 * d)
    c = host.cache(nkvh, hd, 32)
    host.ok("pg_kv_cache_append_dev", host.ctx, c, x, x, 32)             # (room for 64)
    host.ok("pg_kv_cache_rollback_to", c, 64 - seq)
    host.ok("pg_llama_block_forward_dev", host.ctx, b, x, seq, c, out)   # every buffer of the step exists now; the cache is full
    assert host.lib.pg_kv_cache_len(c) == host.lib.pg_kv_cache_capacity(c) == 64
    host.lib.pg_kv_cache_free(host.ctx, host.cache(nkvh, hd, 128))
    st, recorded, whole = host.captured("pg_llama_block_forward_dev", host.ctx, b, x, seq, c, out)
    assert st == 2 and recorded == 0 and whole
    assert host.lib.pg_kv_cache_len(c) == 64
    host.ok("pg_llama_block_forward_dev", host.ctx, b, x, seq, c, out)
    assert host.lib.pg_kv_cache_capacity(c) == 128
    host.ok("pg_kv_cache_rollback_to", c, 64)
    st, recorded, whole = host.captured("pg_llama_block_forward_dev", host.ctx, b, x, seq, c, out)
    assert st == 0 and recorded > 0 and whole
    host.lib.pg_kv_cache_free(host.ctx, c)
    host.lib.pg_llama_block_free(host.ctx, b)


def test_coded_cache_append_that_cuts_a_chunk_is_refused_by_a_capture(host):
    heads, hd = 2, 64
    c = host.new("pg_huffman_kv_cache_create", host.ctx, heads, hd, 32, 32)
    rows = host.alloc(heads * hd * 64)
    for tokens in (31, 1, 31):                                          # 63 tokens: one chunk a side, 31 in the window
        host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, tokens)
    assert host.lib.pg_huffman_kv_cache_num_chunks(c) == 1
    st, recorded, whole = host.captured("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, 1)
    assert st == 2 and recorded == 0 and whole
    assert host.lib.pg_huffman_kv_cache_len(c) == 63
    host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, 1)
    assert host.lib.pg_huffman_kv_cache_num_chunks(c) == 2
    host.lib.pg_huffman_kv_cache_free(host.ctx, c)


def coded_cache(host, heads=8, hd=128, tokens=256, pieces=2):
    """A coded cache that has cut a chunk a side per piece, and the rows of another."""
    c = host.new("pg_huffman_kv_cache_create", host.ctx, heads, hd, tokens, tokens)
    rows = host.alloc(heads * hd * 2 * tokens)
    for _ in range(pieces):
        host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, tokens)
    return c, rows


@pytest.mark.parametrize("mallocs,news", [(n, NO_LIMIT) for n in range(6)] + [(NO_LIMIT, n) for n in range(3)])
@pytest.mark.parametrize("was,now", [(100000, 120000), (100000, 100000), (100000, 5000)])
def test_append_that_runs_out_of_memory_leaves_the_coded_cache_whole(host, mallocs, news, was, now):
    """Every allocation of an append that cuts a chunk fails in turn.  What failed has moved nothing: the only encoder
    launches that carry the window's move are those that do nothing where streams do not suit their rooms, and these
    did not.  The next append cuts what this one could not."""
    host.lib.pghost_stream_bytes(was, was)
    c, rows = coded_cache(host)
    host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, 255)
    drained = host.alloc(1)                                              # (an allocation that fails empties the pool)
    host.lib.pghost_limit(host.lib.pghost_used())
    assert host.lib.pg_dev_alloc(host.ctx, 1 << 20, C.byref(C.c_void_p())) == 3
    host.lib.pghost_limit(NO_LIMIT)
    host.lib.pghost_stream_bytes(now, now)
    host.lib.pghost_clear_launches()
    host.lib.pghost_fail_after(mallocs, news)
    st = host.lib.pg_huffman_kv_cache_append_dev(host.ctx, c, rows, rows, 2)
    host.lib.pghost_fail_after(NO_LIMIT, NO_LIMIT)
    shape = lambda: (host.lib.pg_huffman_kv_cache_len(c), host.lib.pg_huffman_kv_cache_compressed_len(c), host.lib.pg_huffman_kv_cache_num_chunks(c))
    encoders = [name for name, _ in host.launches() if "kv_encode_kernel" in name]
    if st == 0:
        assert shape() == (769, 768, 3)
    else:
        assert st == 3 and shape()[1:] == (512, 2)
        assert shape()[0] in (767, 769)                                  # (767: there was no room for the new rows)
        assert all("kv_encode_kernelILb1E" in name for name in encoders) and (now != was or not encoders), encoders
        n = 769 - shape()[0]
        host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, n)
        if n == 0:
            host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, 1)
        assert shape()[1:] == (768, 3)
    if (mallocs, news) == (0, NO_LIMIT) or news == 0:
        assert st == 3                                                   # (the test does reach failures)
    host.lib.pg_huffman_kv_cache_free(host.ctx, c)
    host.ok("pg_dev_free", host.ctx, drained)


def test_append_that_fits_is_taken_where_a_guess_would_not(host):
    """After streams of 100000 bytes, two of 5000 with memory for them, but not for two like the last."""
    host.lib.pghost_stream_bytes(100000, 100000)
    c, rows = coded_cache(host)
    host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, 255)
    host.lib.pghost_stream_bytes(5000, 5000)
    host.lib.pghost_limit(host.lib.pghost_used())
    assert host.lib.pg_dev_alloc(host.ctx, 1 << 20, C.byref(C.c_void_p())) == 3   # (the pool is empty now)
    host.lib.pghost_limit(host.lib.pghost_used() + 120000)
    host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, 1)
    assert host.lib.pg_huffman_kv_cache_num_chunks(c) == 3
    host.lib.pg_huffman_kv_cache_free(host.ctx, c)


@pytest.mark.parametrize("first,then", [((100000, 100000), (5000, 5000)), ((30000, 220000), (30000, 220000)), ((5000, 5000), (100000, 100000)),
                                        ((100000, 100000), (97500, 97500)), ((100000, 100000), (99000, 101500)), ((40000, 200000), (39000, 190000))])
def test_coded_chunks_take_the_memory_their_streams_need(host, first, then):
    """Streams of one length, then of another, the sides' of their own: a batch holds at most 1 / 32 more than scales, tables,
    index and streams (and the step of the allocations: a sixteenth of a power of two)."""
    heads, hd, tokens = 8, 128, 256
    host.lib.pghost_stream_bytes(*first)
    c, rows = coded_cache(host, heads, hd, tokens)
    host.lib.pghost_stream_bytes(*then)
    total = heads * hd * tokens
    chunk = lambda b: 256 + 256 + 8192 + (total // 4096 + 1) * 8 + total // 64 * 2 + b + 512
    for n in range(3):
        drained = host.lib.pghost_used()
        host.lib.pghost_limit(drained)
        assert host.lib.pg_dev_alloc(host.ctx, 1 << 30, C.byref(C.c_void_p())) == 3
        host.lib.pghost_limit(NO_LIMIT)
        before = host.lib.pghost_used()
        host.lib.pghost_clear_launches()
        host.ok("pg_huffman_kv_cache_append_dev", host.ctx, c, rows, rows, tokens)
        encoders = [name for name, _ in host.launches() if "kv_encode_kernel" in name]
        assert len(encoders) in (1, 2) and "ILb1E" in encoders[0], encoders
        host.lib.pghost_limit(host.lib.pghost_used())                    # (a guess that did not suit lies in the pool)
        assert host.lib.pg_dev_alloc(host.ctx, 1 << 30, C.byref(C.c_void_p())) == 3
        host.lib.pghost_limit(NO_LIMIT)
        taken, need = host.lib.pghost_used() - before, sum(chunk(b) for b in then)
        assert taken <= need * (1 + 1 / 32) * (1 + 1 / 8), (taken, need)
        assert n == 0 or len(encoders) == 1                              # and like the last, one launch
    host.lib.pg_huffman_kv_cache_free(host.ctx, c)


def f16_route(host, typ, m, n, k):
    """Whether a product of m rows over an [n, k] tensor runs on the f16 matrix cores."""
    w = host.new("pg_gguf_upload", host.ctx, bytes(n * k // 32 * {2: 18, 3: 20, 8: 34}[typ]), typ, n, k)
    x, y = host.alloc(m * k), host.alloc(m * n)
    host.lib.pghost_clear_launches()
    host.ok("pg_gguf_matmul_dev", host.ctx, x, m, w, y)
    host.lib.pg_gguf_free(host.ctx, w)
    for p in (x, y):
        host.ok("pg_dev_free", host.ctx, p)
    return any("gguf_hmm_kernel" in name for name, _ in host.launches())


@pytest.mark.parametrize("typ", [2, 3, 8])
def test_products_of_the_f16_route_stay_there(host, typ):
    """From 96 rows and 18 G (Q8_0: 24 G) multiply-adds on, a product always ran with its activations in f16 planes (2^-22
    of a row's largest value): no estimate may hand it to the int8 block route (2^-16 of a block's)."""
    least = 2.4e10 if typ == 8 else 1.8e10
    for k, n in ((4096, 22016), (4096, 14336), (2048, 11008), (14336, 4096), (8192, 8200), (1024, 32000), (13312, 1029), (6528, 32772)):
        first = max(96, int(-(-least // (n * k))))
        for m in sorted({first, first + 1, first + 10, first + 21, first + 26, first + 45}):
            if m * n * k <= 4e10:
                assert f16_route(host, typ, m, n, k), (typ, m, n, k)


@pytest.mark.parametrize("typ,m,k,n,f16", [
    (2, 60, 14336, 14336, True), (2, 640, 6656, 2570, True), (8, 583, 4736, 4313, True), (8, 130, 5632, 9000, True), (3, 120, 8192, 6000, True),   # by their time
    (2, 48, 14336, 14336, False), (2, 72, 2048, 16384, False), (2, 200, 2048, 16384, False), (8, 150, 2048, 8192, False), (3, 200, 4096, 4096, False),
    (8, 278, 4096, 14438, True), (2, 169, 7616, 11455, True), (2, 140, 6144, 13965, True), (8, 267, 5184, 11881, True), (8, 886, 3904, 4478, True),  # held
])
def test_which_products_run_on_the_f16_matrix_cores(host, typ, m, k, n, f16):
    """Both sides of the line between the routes, and products that keep their finer activations though the int8 route is estimated to be as fast."""
    assert f16_route(host, typ, m, n, k) == f16


def dequant_i8_call(host, m, k, n):
    """The kernels of one W8A32 product and the scratch it made the context take."""
    w = host.alloc(k * n)
    q = host.new("pg_qtensor_from_f32_dev", host.ctx, w, k, n)
    host.ok("pg_dev_free", host.ctx, w)
    x, y = host.alloc(m * k), host.alloc(m * n)
    host.lib.pghost_clear_launches()
    before = host.lib.pghost_used()
    host.ok("pg_matmul_dequant_i8_dev", host.ctx, x, m, k, q, y)
    taken = host.lib.pghost_used() - before
    for p in (x, y):
        host.ok("pg_dev_free", host.ctx, p)
    host.lib.pg_qtensor_free(host.ctx, q)
    return [name for name, _ in host.launches()], taken


@pytest.mark.parametrize("m", [1, 16, 32, 33, 100, 191, 257, 383])
@pytest.mark.parametrize("n", [45825, 50257, 65536, 128256])
def test_w8a32_over_wide_weights_is_one_launch_in_the_planes_scratch(host, m, n):
    """A vocabulary's columns: few 256-row tiles of many columns are still few rows.  One launch after the rows' digits, and
    no scratch beyond the three planes (the accumulator planes of the stacked form are 8 bytes per padded row and column)."""
    k = 1024
    names, taken = dequant_i8_call(host, m, k, n)
    assert len(names) == 2 and ("skinny" if m <= 32 else "gemm_w8a8_kernel") in names[1], names
    m_pad = -(-m // 256) * 256
    assert taken <= 1.25 * 3 * (m_pad * k + 4 * m_pad) + (2 << 20), taken


@pytest.mark.parametrize("m,k,n", [(192, 256, 46080), (191, 256, 46080), (384, 256, 23040), (2048, 256, 5888), (192, 256, 98049), (1000, 4096, 4096), (2048, 4096, 14336)])
def test_w8a32_large_products_are_one_launch(host, m, k, n):
    """Products that fill the part with 256x256 tiles that are mostly rows: as three launches over stacked planes 69 us where one takes 22
    (192 x 256 -> 46080), 382 : 293 (2048 x 4096 -> 14336), 115 : 51 (1000 x 4096 -> 4096)."""
    names, _ = dequant_i8_call(host, m, k, n)
    assert len(names) == 2, names


@pytest.mark.parametrize("m,k,stacked", [(8192, 130048, False), (8192, 130049, True), (7936, 132104, False), (8193, 130048, True)])
def test_w8a32_products_beyond_one_launchs_offsets_stack_their_low_planes(host, m, k, stacked):
    """Both sides of the line: two planes of the padded rows and 128 rows of weights within 2^31 bytes."""
    names, _ = dequant_i8_call(host, m, k, 64)
    assert len(names) == (3 if stacked else 2), names


def test_memory_running_out_empties_the_pool_for_every_allocation(host):
    """64 MB lie in the pool (a key/value cache's two planes); with 16 MB of device memory left, whatever needs more
    than that gets it: the workspace, a block's chain and arena, weights, temporaries, the caller's own allocations."""
    mb = 1 << 20
    d, nqh, nkvh, hd, ffn, seq = 256, 4, 2, 64, 8192, 400
    shapes = [(nqh * hd, d), (nkvh * hd, d), (nkvh * hd, d), (d, nqh * hd), (ffn, d), (ffn, d), (d, ffn)]
    ws = [host.gguf(n, k) for n, k in shapes]
    b = host.new("pg_llama_block_create", host.ctx, d, nqh, nkvh, hd, ffn, 512, 10000.0, 1e-5)
    norm = np.ones(d, np.float32)
    host.ok("pg_llama_block_set_weights", host.ctx, b, *ws, norm.ctypes.data, norm.ctypes.data)
    c, x = host.cache(nkvh, hd, 32), host.alloc(seq * d)
    k, n, m = 4096, 8192, 64
    wf, y, xq = host.alloc(k * n), host.alloc(m * n), host.alloc(2048 * k)
    q = host.new("pg_qtensor_from_f32_dev", host.ctx, wf, k, 64)
    i8, scales = np.zeros(k * n, np.int8), np.ones(n, np.float32)
    out = np.zeros(seq * d, np.float32)

    def upload():
        host.lib.pg_qtensor_free(host.ctx, host.new("pg_qtensor_upload", host.ctx, i8.ctypes.data, scales.ctypes.data, k, n))

    def rows():
        big = np.zeros(6 * mb, np.float32)
        host.ok("pg_rmsnorm", host.ctx, big.ctypes.data, 6 * mb // d, d, norm.ctypes.data, 1e-5, big.ctypes.data)

    for what, use in (("workspace", lambda: host.ok("pg_matmul_dequant_i8_dev", host.ctx, xq, 2048, k, q, y)),
                      ("block step", lambda: host.ok("pg_llama_block_forward_dev", host.ctx, b, x, seq, c, x)),
                      ("weights", upload), ("temporaries", rows),
                      ("a caller's", lambda: host.ok("pg_dev_free", host.ctx, host.alloc(8 * mb)))):
        planes = host.cache(8, 128, 8192)
        used = host.lib.pghost_used()
        host.lib.pg_kv_cache_free(host.ctx, planes)
        assert host.lib.pghost_used() == used                     # (64 MB in the pool now)
        host.lib.pghost_limit(used + 16 * mb)
        use()
        host.lib.pghost_limit(C.c_size_t(-1).value)
        assert host.lib.pghost_used() < used + 16 * mb, what
    host.lib.pg_kv_cache_free(host.ctx, c)
    host.lib.pg_llama_block_free(host.ctx, b)


@pytest.mark.parametrize("users", ["a", "ab", "aba", "abab"])
def test_memory_another_context_has_used_is_not_pooled(host, users):
    """A cache and a coded cache used on two contexts' streams in turn, from the first of which they are freed: what only
    the one context used goes to its pool, everything else to hipFree, which waits for both streams -- chunks and tables
    made after the window was shared among it."""
    other = host.new("pg_ctx_create", 0, None)
    ctx = {"a": host.ctx, "b": other}
    heads, hd = 2, 64
    rows, out = host.alloc(heads * hd * 256), host.alloc(heads * hd * 256)
    plain = host.new("pg_kv_cache_create", host.ctx, heads, hd)
    coded = host.new("pg_huffman_kv_cache_create", host.ctx, heads, hd, 32, 32)
    for u in users:
        host.ok("pg_kv_cache_append_dev", ctx[u], plain, rows, rows, 8)       # (room for 32: it never grows)
        host.ok("pg_huffman_kv_cache_append_dev", ctx[u], coded, rows, rows, 33)   # a chunk each
    host.ok("pg_huffman_kv_cache_get_kv_dev", host.ctx, coded, out, out)
    for cache, free, blocks in ((plain, "pg_kv_cache_free", 2), (coded, "pg_huffman_kv_cache_free", 3 + len(users))):
        before = host.lib.pghost_frees()
        getattr(host.lib, free)(host.ctx, cache)
        freed = host.lib.pghost_frees() - before
        if users == "a":
            assert freed == 0                                                 # all of it pooled
        elif cache is plain:
            assert freed == 2
        else:
            # two planes of the window, the table, and the chunks: a reads b's, and b's appends follow a's first
            own_after = 1 if users == "aba" else 0                            # the chunk that a cut after b's last use
            assert freed == blocks - own_after, (freed, blocks)
    host.lib.pg_ctx_destroy(other)


@pytest.mark.parametrize("m,k,n,tiles", [
    (197, 1024, 4096, ["64ELi64ELi128ELi3ELi4ELi2E"]),                             # 10.3 us on eight wavefronts; on four 11.1, 32x128 10.8
    (356, 4096, 14336, ["64ELi128E"]),                                             # 78; 64x256 87
    (1000, 4096, 4096, ["64ELi256E"]),                                             # 51; 64x128 59, 128x128 58
    (311, 2048, 32000, ["64ELi128E", "64ELi256E"]),                                # 75 and 74; 32x128 86
    (155, 1024, 103918, ["64ELi128E", "32ELi128ELi128ELi2E", "64ELi256E"]),        # 89, 89 and 90; the next 107
    (888, 11222, 4096, ["64ELi256E"]),                                             # 123; 64x128 132
    (334, 104, 42211, ["128ELi128ELi128ELi2ELi4ELi4E"]),                           # 28.7 on sixteen wavefronts; on eight 42.0, 64x128 33.4
    (120, 111, 62971, ["128ELi128ELi128ELi2ELi4ELi4E"]),                           # 17.4; 24.7, 20.4
    (467, 8337, 534, ["32ELi64E"]),                                                # 37.2; 64x64 42.2
])
def test_w8a32_tile_is_the_one_that_took_least(host, m, k, n, tiles):
    """Or one within 2 % of it (us, beside each)."""
    names, _ = dequant_i8_call(host, m, k, n)
    assert len(names) == 2 and any("gemm_w8a8_kernelILi" + t in names[1] for t in tiles), names


def int8_call(host, m, k, ns):
    """The kernels of one W8A8 product over one weight or several."""
    qs = []
    for n in ns:
        w = host.alloc(k * n)
        qs.append(host.new("pg_qtensor_from_f32_dev", host.ctx, w, k, n))
        host.ok("pg_dev_free", host.ctx, w)
    x, outs = host.alloc(m * k), [host.alloc(m * n) for n in ns]
    host.lib.pghost_clear_launches()
    if len(ns) == 1:
        host.ok("pg_matmul_quantized_dev", host.ctx, x, m, k, qs[0], outs[0], None)
    else:
        tab = lambda of: (C.c_void_p * len(of))(*[p.value for p in of])
        host.ok("pg_matmul_quantized_multi_dev", host.ctx, x, m, k, tab(qs), len(ns), tab(outs))
    for p in [x] + outs:
        host.ok("pg_dev_free", host.ctx, p)
    for q in qs:
        host.lib.pg_qtensor_free(host.ctx, q)
    return [name for name, _ in host.launches()]


def tile(bm, bn):
    return "gemm_w8a8_kernelILi%dELi%dE" % (bm, bn)


def rows_in_groups(mb, nb, nw, nst):
    return "gemm_w8a8_skinny_kernelILi%dELi%dELi%dELi%dELb0ELb1E" % (mb, nb, nw, nst)


@pytest.mark.parametrize("m,k,ns,kernel,finish", [
    (225, 4026, [1099], rows_in_groups(3, 2, 8, 2), False),           # 12.6 us; groups of 48 rows, a weight tile each, 17.4: 69 weight tiles x 5 on 8 XCDs
    (110, 5660, [1350], rows_in_groups(2, 2, 8, 2), False),           # 12.3; 16.3
    (197, 6464, [298, 507], rows_in_groups(2, 2, 8, 2), False),       # 13.2; 18.5
    (200, 10240, [50257], tile(256, 256), False),                     # 165; 197 on 128x64
    (111, 7102, [49915], tile(128, 256), False),                      # 87; 120
    (100, 4096, [50257], tile(128, 256), False),                      # 56; 70
    (40, 1024, [50257], tile(64, 64), False),                         # 19.5; all rows in a workgroup 29.6
    (62, 5302, [14499], tile(64, 64), False),                         # 22.7; 28.4
    (163, 12022, [6319], tile(128, 128), True),                       # 43.1; 58.2 on 64x64
    (132, 9671, [2828, 7938], tile(64, 64), False),                   # 50; 70 with one apart
    (288, 117, [97561], tile(256, 256), False),                       # 32.5; 47.4 on 64x64
    (544, 71, [49642], tile(128, 256), False),                        # 31.1; 43.1 on 64x64
    (530, 631, [65280], tile(256, 256), False),                       # 71.7; 89.4 on 128x256
    (1779, 512, [6406], tile(256, 192), False),                       # 20.5; 26.0 on 256x128
    (184, 11725, [6400], tile(128, 128), True),                       # 45.7; 59.0 on 64x64
    (99, 9010, [1029], rows_in_groups(3, 1, 8, 2), False),            # 15.9; 20.8 on 64x64, K split
])
def test_int8_product_of_some_rows_takes_a_kernel_that_was_clearly_faster(host, m, k, ns, kernel, finish):
    """Products of which another kernel took at least a tenth longer than this one (us, both sides beside them)."""
    names = int8_call(host, m, k, ns)
    assert kernel in names[1] and len(names) == 2 + finish and ("splitk_finish" in names[-1]) == finish, names


@pytest.mark.parametrize("m,k,n,resident", [(195, 15812, 3090, 1), (200, 15888, 3081, 1), (33, 13376, 2060, 2), (34, 13823, 2079, 2), (65, 11004, 8720, 1)])
def test_int8_runs_of_k_are_as_many_as_an_xcd_has_places(host, m, k, n, resident):
    """An XCD has all runs of every eighth tile; counted over the part, 50 tiles in five runs are 35 workgroups for its 32 CUs."""
    names = int8_call(host, m, k, [n])
    assert len(names) == 3 and "splitk_finish" in names[2], names
    tiles, runs = host.launches()[1][1][:2]
    assert tiles % 8 == 0 and 2 <= runs and tiles // 8 * runs <= 32 * resident, (tiles, runs)


@pytest.mark.parametrize("m,k,n,kernel", H.INT8_ROUTES)
def test_int8_products_run_on_the_kernels_that_they_are_tested_on(host, m, k, n, kernel):
    """What the results of these products are compared for (test_gpu_quant.py): every kernel from 33 rows on."""
    names = int8_call(host, m, k, [n])
    assert kernel in names[1] and len(names) == (3 if (m, k, n) in H.INT8_SPLIT else 2), names


@pytest.mark.parametrize("m,k,n,kernel", H.W8A32_ROUTES)
def test_w8a32_products_run_on_the_kernels_that_they_are_tested_on(host, m, k, n, kernel):
    names, _ = dequant_i8_call(host, m, k, n)
    assert kernel in names[1] and len(names) == 2, names


def test_the_tested_int8_kernels_are_all_there_are():
    assert len({r[3] for r in H.INT8_ROUTES}) == 8 + 8 and len({r[3] for r in H.W8A32_ROUTES}) == 10   # (256x256: the prefill shapes)


@pytest.mark.parametrize("code,bm,bn", [(1, 64, 64), (2, 256, 256), (3, 128, 256), (4, 128, 64), (5, 128, 128), (6, 256, 256), (7, 256, 256), (8, 256, 256)])
def test_w8a32_last_pass_by_tile_override(host, code, bm, bn):
    host.ok("pg_gemm_w8a8_force_tile", host.ctx, code)
    names, _ = dequant_i8_call(host, 2048, 128, 5888)
    host.ok("pg_gemm_w8a8_force_tile", host.ctx, 0)
    assert len(names) == 3 and "gemm_w8a8_kernelILi%dELi%dE" % (bm, bn) in names[2] and "ELb0ELb1ELi1E" in names[2], names


@pytest.mark.parametrize("m,k,n,kernel", [(467, 8337, 534, "kernelILi32ELi64E"), (257, 2717, 783, "kernelILi32ELi64E"), (56, 8914, 7775, "kernelILi32ELi64E")])
def test_w8a32_groups_of_rows_are_counted_by_xcd(host, m, k, n, kernel):
    """34.1 us against 58.6 in groups of 32 rows, whose 17 weight tiles x 15 groups are up to 45 workgroups for an XCD's 32
    CUs; 16.5 against 20.4.  (The last one by the margin: 30.7 against 36.3 on 64x64.)"""
    names, _ = dequant_i8_call(host, m, k, n)
    assert kernel in names[1], names


@pytest.mark.parametrize("n,k,m,runs", [
    (70, 832, 65, True), (972, 1216, 1008, True), (2048, 832, 512, True), (2282, 9760, 70, True), (3072, 1088, 512, True), (3072, 14336, 1024, True),
    (70, 768, 65, False), (2049, 1024, 512, False), (3073, 1088, 512, False), (13241, 960, 171, False), (5268, 1184, 413, False), (2895, 864, 738, False),
    (6144, 4096, 512, False), (6144, 4160, 513, False), (14336, 512, 200, False),
])
def test_q4_1_offsets_in_runs_where_that_is_shorter(host, n, k, m, runs):
    """Both sides of each line between four runs of a tile's blocks and four tiles side by side.  171 x 960 -> 13241 takes 37.0 us side by side and
    41.3 in runs, 413 x 1184 -> 5268 37.0 and 40.0, 738 x 864 -> 2895 37.5 and 41.4."""
    w = host.new("pg_gguf_upload", host.ctx, bytes(H.pack_q4_1(np.zeros(n * k, np.float32))), 3, n, k)
    x, y = host.alloc(m * k), host.alloc(m * n)
    host.ok("pg_gguf_hmm_force", host.ctx, 1)
    host.lib.pghost_clear_launches()
    host.ok("pg_gguf_matmul_dev", host.ctx, x, m, w, y)
    names = [name for name, _ in host.launches() if "q41_offset" in name]
    assert len(names) == 1 and ("q41_offset_mfma_kernelILb%dE" % runs) in names[0], names
    host.ok("pg_gguf_hmm_force", host.ctx, 0)
    for p in (x, y):
        host.ok("pg_dev_free", host.ctx, p)
    host.lib.pg_gguf_free(host.ctx, w)


def same_call_captured(host, name, *args):
    """A call that has run once at its shape is captured whole, as launches alone."""
    host.ok(name, host.ctx, *args)
    st, recorded, whole = host.captured(name, host.ctx, *args)
    assert st == 0 and whole and recorded > 0 and host.lib.pghost_copied() == 0, (name, st, recorded, whole, host.lib.pghost_copied(), host.lib.pg_last_error())


ROWS = [1, 2, 3, 5, 8, 9, 16, 17, 33, 64, 65, 97, 150, 200, 300, 700]


@pytest.mark.parametrize("typ", [2, 3, 8])
@pytest.mark.parametrize("n,k", [(4096, 4096), (1000, 1024), (1029, 6656), (300, 96)])
def test_block_products_are_captured_after_one_eager_call(host, typ, n, k):
    w = host.new("pg_gguf_upload", host.ctx, bytes(n * k // 32 * {2: 18, 3: 20, 8: 34}[typ]), typ, n, k)
    x, y = host.alloc(max(ROWS) * k), host.alloc(max(ROWS) * n)
    for m in ROWS:
        same_call_captured(host, "pg_gguf_matmul_dev", x, m, w, y)


@pytest.mark.parametrize("n,k", [(4096, 1024), (50257, 256), (300, 4096)])
def test_int8_products_are_captured_after_one_eager_call(host, n, k):
    w = host.alloc(n * k)
    q = host.new("pg_qtensor_from_f32_dev", host.ctx, w, k, n)
    x, y = host.alloc(max(ROWS) * k), host.alloc(max(ROWS) * n)
    for m in ROWS:
        same_call_captured(host, "pg_matmul_quantized_dev", x, m, k, q, y, None)
        same_call_captured(host, "pg_matmul_dequant_i8_dev", x, m, k, q, y)


@pytest.mark.parametrize("call", ["pg_matmul_quantized_dev", "pg_matmul_dequant_i8_dev"])
@pytest.mark.parametrize("n,k", [(643, 8192), (832, 7055), (756, 5127), (134, 8143), (4096, 14336), (2373, 6563), (289, 12805), (534, 8337), (50257, 256)])
def test_int8_products_of_fewer_rows_need_no_more_scratch(host, call, n, k):
    """A program that has run its largest batch captures any smaller one: K is split over workgroups, with partial sums in the scratch, for some
    numbers of rows only (8192 -> 643: 488, but not 1024), and the workspace does not grow for them.  Nor does it grow eagerly, which would free
    the one that an earlier graph writes."""
    w = host.alloc(n * k)
    q = host.new("pg_qtensor_from_f32_dev", host.ctx, w, k, n)
    rows = sorted({1, 5, 33, 48, 62, 64, 65, 97, 129, 200, 257, 286, 320, 321, 385, 467, 488, 513, 645, 700, 701, 900, 1024, 2048}, reverse=True)
    x, y = host.alloc(rows[0] * k), host.alloc(rows[0] * n)
    args = lambda m: (x, m, k, q, y) + ((None,) if call == "pg_matmul_quantized_dev" else ())
    for i, largest in enumerate(rows):
        ctx = host.new("pg_ctx_create", 0, None)
        host.ok(call, ctx, *args(largest))
        used = host.lib.pghost_used()
        for m in rows[i + 1:]:
            host.lib.pghost_begin_capture(host.stream(ctx))
            st = getattr(host.lib, call)(ctx, *args(m))
            assert host.lib.pghost_end_capture(host.stream(ctx)) and st == 0, (largest, m, host.lib.pg_last_error())
            host.ok(call, ctx, *args(m))
            assert host.lib.pghost_used() == used, (largest, m)
        host.lib.pg_ctx_destroy(ctx)
    host.lib.pg_qtensor_free(host.ctx, q)


SPLIT_CALLS = [("pg_matmul_quantized_dev", 488, 643, 8192, "splitk_finish_kernel"), ("pg_matmul_dequant_i8_dev", 286, 832, 7055, "splitk_finish_w8a32")]


@pytest.mark.parametrize("call,m,n,k,finish", SPLIT_CALLS)
def test_int8_products_are_captured_whole_where_the_scratch_has_no_room_to_split_k(host, call, m, n, k, finish):
    """The partial sums are no reason to refuse a capture: whatever eager call has left room for the rows, K is split where its planes find
    room behind them and walked whole where they do not (integer sums: the same bits).  Only rows without room are refused."""
    w = host.alloc(n * k)
    q = host.new("pg_qtensor_from_f32_dev", host.ctx, w, k, n)
    few = host.new("pg_qtensor_from_f32_dev", host.ctx, host.alloc(8 * 4096), 4096, 8)
    x, y = host.alloc(2048 * 4096), host.alloc(2048 * n)
    tail = (None,) if call == "pg_matmul_quantized_dev" else ()
    seen = []
    for rows in range(0, 2049, 256):     # of another weight, whose rows alone size the scratch
        ctx = host.new("pg_ctx_create", 0, None)
        before = host.lib.pghost_used()
        if rows:
            host.ok("pg_matmul_dequant_i8_dev", ctx, x, rows, 4096, few, y)
        arena = host.lib.pghost_used() - before
        host.lib.pghost_clear_launches()
        host.lib.pghost_begin_capture(host.stream(ctx))
        st = getattr(host.lib, call)(ctx, x, m, k, q, y, *tail)
        assert host.lib.pghost_end_capture(host.stream(ctx)) == (st == 0)
        names = [name for name, _ in host.launches()]
        seen.append("refused" if st else "split" if finish in names[-1] else "whole")
        assert host.lib.pghost_used() - before == arena
        host.lib.pg_ctx_destroy(ctx)
    assert seen[0] == "refused" and seen[-1] == "split" and "whole" in seen, seen
    assert seen == sorted(seen, key=["refused", "whole", "split"].index), seen
    for t in (q, few):
        host.lib.pg_qtensor_free(host.ctx, t)


@pytest.mark.parametrize("call,m,n,k,finish", SPLIT_CALLS)
def test_int8_products_do_without_the_room_to_split_k_where_memory_has_run_out(host, call, m, n, k, finish):
    w = host.alloc(n * k)
    q = host.new("pg_qtensor_from_f32_dev", host.ctx, w, k, n)
    x, y = host.alloc(m * k), host.alloc(m * n)
    tail = (None,) if call == "pg_matmul_quantized_dev" else ()
    k_pad, m_pad = (k + 127) // 128 * 128, (m + 255) // 256 * 256
    rows = m_pad * k_pad * (1 if tail else 3)
    used, seen = host.lib.pghost_used(), []
    for free in (rows // 2, rows * 5 // 4 + (2 << 20), rows * 5 // 4 + (80 << 20)):
        ctx = host.new("pg_ctx_create", 0, None)
        host.lib.pghost_limit(used + free)
        host.lib.pghost_clear_launches()
        st = getattr(host.lib, call)(ctx, x, m, k, q, y, *tail)
        host.lib.pghost_limit(NO_LIMIT)
        names = [name for name, _ in host.launches()]
        seen.append("refused" if st else "split" if finish in names[-1] else "whole")
        host.lib.pg_ctx_destroy(ctx)
    assert seen == ["refused", "whole", "split"], seen
    host.lib.pg_qtensor_free(host.ctx, q)


def test_expert_layers_are_captured_after_one_eager_call(host):
    d, ffn, E, k = 256, 512, 8, 2
    tab = lambda n_out, k_in: (C.c_void_p * E)(*[host.new("pg_gguf_upload", host.ctx, bytes(n_out * k_in // 32 * 34), 8, n_out, k_in).value for _ in range(E)])
    gate, up, down = (C.cast(t, C.POINTER(C.c_void_p)) for t in (tab(ffn, d), tab(ffn, d), tab(d, ffn)))
    codes, scales, bias = np.zeros(2 * ffn * d // 2, np.uint8), np.zeros(2 * ffn * d // 32, np.uint8), np.zeros(2 * ffn, np.float32)
    p = lambda a: a.ctypes.data
    ex = (C.c_void_p * E)(*[host.new("pg_mxfp4_expert_create", host.ctx, d, ffn, 1.702, 7.0, p(codes), p(scales), p(bias), p(codes), p(scales), p(bias)).value
                            for _ in range(E)])
    x, logits, out = host.alloc(700 * d), host.alloc(700 * E), host.alloc(700 * d)
    idx, wt = host.alloc(700 * k), host.alloc(700 * k)
    for T in ROWS:
        same_call_captured(host, "pg_moe_ffn_dev", x, T, logits, E, k, gate, up, down, 0, out)
        same_call_captured(host, "pg_mxfp4_moe_ffn_routed_dev", x, T, idx, wt, k, C.cast(ex, C.POINTER(C.c_void_p)), E, out)


@pytest.mark.parametrize("typ,d,ffn", [(2, 256, 512), (8, 1024, 2048), (3, 256, 512)])
def test_block_steps_are_captured_after_one_eager_call(host, typ, d, ffn):
    nqh, nkvh, hd = 4, 2, 64
    shapes = [(nqh * hd, d), (nkvh * hd, d), (nkvh * hd, d), (d, nqh * hd), (ffn, d), (ffn, d), (d, ffn)]
    ws = [host.new("pg_gguf_upload", host.ctx, bytes(n * k // 32 * {2: 18, 3: 20, 8: 34}[typ]), typ, n, k) for n, k in shapes]
    b = host.new("pg_llama_block_create", host.ctx, d, nqh, nkvh, hd, ffn, 2048, 10000.0, 1e-5)
    norm = np.ones(d, np.float32)
    host.ok("pg_llama_block_set_weights", host.ctx, b, *ws, norm.ctypes.data, norm.ctypes.data)
    x, out = host.alloc(700 * d), host.alloc(700 * d)
    c = host.cache(nkvh, hd, 1500)
    for seq in ROWS:
        for at in (0, 700):
            host.ok("pg_kv_cache_rollback_to", c, min(at, host.lib.pg_kv_cache_len(c)))
            host.ok("pg_llama_block_forward_dev", host.ctx, b, x, seq, c, out)
            host.ok("pg_kv_cache_rollback_to", c, host.lib.pg_kv_cache_len(c) - seq)
            st, recorded, whole = host.captured("pg_llama_block_forward_dev", host.ctx, b, x, seq, c, out)
            assert st == 0 and whole and recorded > 0 and host.lib.pghost_copied() == 0, (seq, at, host.lib.pg_last_error())
    host.lib.pg_kv_cache_free(host.ctx, c)
    host.lib.pg_llama_block_free(host.ctx, b)
