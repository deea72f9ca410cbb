"""Shared test helpers: fixture loading, deterministic generators the reference's own
tests use, and block packers for synthetic GGUF tensors."""
import os
import struct

import numpy as np

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def load_fixture(name):
    """[ndim u32][shape u32...][f32 data]  (reference: tests/pytorch_parity.rs:16-39)."""
    buf = open(os.path.join(GOLDEN, name), "rb").read()
    ndim = struct.unpack_from("<I", buf, 0)[0]
    shape = struct.unpack_from(f"<{ndim}I", buf, 4)
    data = np.frombuffer(buf, np.float32, int(np.prod(shape)), 4 + 4 * ndim)
    return data.reshape(shape).copy()


def lcg_data(n, seed):
    """tests/huffman_parity.rs:7-16: s = s*1103515245 + 12345 (u32); f = s/u32::MAX*2 - 1."""
    out = np.empty(n, np.float32)
    s = seed & 0xFFFFFFFF
    umax = np.float32(4294967295.0)
    for i in range(n):
        s = (s * 1103515245 + 12345) & 0xFFFFFFFF
        out[i] = np.float32(s) / umax * np.float32(2.0) - np.float32(1.0)
    return out


def mod_pattern(n, mul, add, mod, div, sub):
    """((i*mul + add) % mod) as f32 / div - sub  (tests/quant_parity.rs:10-12,40-45)."""
    i = np.arange(n, dtype=np.int64)
    return (((i * mul + add) % mod).astype(np.float32) / np.float32(div) - np.float32(sub)).astype(np.float32)


from peregrine_amd.synth import pack_q4_0, pack_q4_1, pack_q8_0  # noqa: E402,F401


def np_dequant_q4_0(raw, n):
    """Independent NumPy statement of the Q4_0 format (value = (q - 8) * d, interleaved)."""
    b = np.frombuffer(raw, np.uint8)[: n // 32 * 18].reshape(-1, 18)
    d = b[:, 0:2].copy().view(np.float16).astype(np.float32)
    lo = (b[:, 2:] & 15).astype(np.int32) - 8
    hi = (b[:, 2:] >> 4).astype(np.int32) - 8
    out = np.empty((b.shape[0], 32), np.float32)
    out[:, 0::2] = lo.astype(np.float32) * d
    out[:, 1::2] = hi.astype(np.float32) * d
    return out.reshape(-1)


def np_dequant_q8_0(raw, n):
    b = np.frombuffer(raw, np.uint8)[: n // 32 * 34].reshape(-1, 34)
    d = b[:, 0:2].copy().view(np.float16).astype(np.float32)
    q = b[:, 2:].copy().view(np.int8).astype(np.float32)
    return (q * d).reshape(-1)


def assert_close_rel(got, ref, rtol, what=""):
    """|got - ref| <= rtol * max(|ref|, rms(ref)): relative to each element, with the
    vector's RMS as the floor for entries that cancel to near zero."""
    got = np.asarray(got, np.float64).reshape(-1)
    ref = np.asarray(ref, np.float64).reshape(-1)
    assert got.shape == ref.shape, (got.shape, ref.shape)
    assert np.isfinite(got).all(), f"{what}: non-finite output"
    floor = np.sqrt(np.mean(ref * ref)) if ref.size else 0.0
    bound = rtol * np.maximum(np.abs(ref), floor)
    err = np.abs(got - ref)
    worst = int(np.argmax(err - bound)) if ref.size else 0
    assert (err <= bound).all(), (
        f"{what}: element {worst}: got {got[worst]!r}, want {ref[worst]!r}, err {err[worst]:.3e} > {bound[worst]:.3e}")


# ---- a GGUF writer for the container tests (format: reference src/gguf.rs:411-483) ----
GGUF_TYPE_CODES = {"u8": 0, "i8": 1, "u16": 2, "i16": 3, "u32": 4, "i32": 5, "f32": 6, "bool": 7, "str": 8,
                   "arr": 9, "u64": 10, "i64": 11, "f64": 12}
_GGUF_FMT = {"u8": "<B", "i8": "<b", "u16": "<H", "i16": "<h", "u32": "<I", "i32": "<i", "f32": "<f", "bool": "<B",
             "u64": "<Q", "i64": "<q", "f64": "<d"}


def _gguf_str(s):
    import struct
    b = s.encode()
    return struct.pack("<Q", len(b)) + b


def _gguf_value(kind, v):
    import struct
    if kind == "str":
        return _gguf_str(v)
    if kind == "arr":  # v = (element kind, [elements])
        ek, items = v
        return struct.pack("<IQ", GGUF_TYPE_CODES[ek], len(items)) + b"".join(_gguf_value(ek, x) for x in items)
    return struct.pack(_GGUF_FMT[kind], v)


def build_gguf(metadata, tensors, version=3, magic=0x46554747):
    """metadata: list of (key, kind, value); tensors: list of (name, ggml_type, shape_gguf_order, raw_bytes).
    Returns (file bytes, data_start, {name: offset in data section})."""
    import struct
    align = 32
    for key, kind, v in metadata:
        if key == "general.alignment":
            align = int(v)
    head = struct.pack("<IIQQ", magic, version, len(tensors), len(metadata))
    for key, kind, v in metadata:
        head += _gguf_str(key) + struct.pack("<I", GGUF_TYPE_CODES[kind]) + _gguf_value(kind, v)
    offsets, off = {}, 0
    for name, typ, shape, raw in tensors:
        offsets[name] = off
        head += _gguf_str(name) + struct.pack("<I", len(shape)) + b"".join(struct.pack("<Q", d) for d in shape)
        head += struct.pack("<IQ", typ, off)
        off = (off + len(raw) + align - 1) // align * align
    data_start = (len(head) + align - 1) // align * align
    body = bytearray(off)
    for name, typ, shape, raw in tensors:
        body[offsets[name]: offsets[name] + len(raw)] = raw
    return head + b"\0" * (data_start - len(head)) + bytes(body), data_start, offsets


# Small ragged products and the kernel each runs on, by the dispatch's own choice: a name's part, as the compiler spells it.
def _tile(bm, bn, nst):
    return "gemm_w8a8_kernelILi%dELi%dELi128ELi%dE" % (bm, bn, nst)


def _rows(mb, nb, nw, nst, tri):
    return "gemm_w8a8_skinny_kernelILi%dELi%dELi%dELi%dELb%dELb1E" % (mb, nb, nw, nst, tri)


INT8_ROUTES = [
    (410, 69, 4953, _tile(64, 64, 3)), (249, 184, 3406, _tile(64, 64, 4)), (260, 95, 10721, _tile(128, 64, 3)), (200, 3358, 10066, _tile(128, 128, 4)),
    (257, 1191, 11804, _tile(128, 192, 3)), (1117, 478, 6849, _tile(128, 256, 3)), (907, 67, 4767, _tile(256, 128, 3)), (1910, 664, 5893, _tile(256, 192, 2)),
    (36, 12871, 303, _tile(64, 64, 4)), (243, 12127, 17, _tile(64, 64, 4)), (65, 11004, 8720, _tile(128, 128, 4)),                     # K split
    (34, 132, 8294, _rows(2, 1, 2, 2, 0)), (46, 72, 7032, _rows(2, 1, 2, 2, 0)), (85, 259, 2159, _rows(2, 1, 4, 3, 0)), (209, 192, 214, _rows(2, 1, 8, 3, 0)),
    (41, 292, 4200, _rows(2, 2, 4, 2, 0)), (268, 294, 422, _rows(2, 2, 8, 2, 0)), (346, 12805, 289, _rows(3, 1, 8, 2, 0)),
    (109, 513, 2335, _rows(3, 2, 8, 2, 0)), (52, 2329, 4970, _rows(4, 2, 4, 3, 0)),
]
INT8_SPLIT = {(36, 12871, 303), (243, 12127, 17), (65, 11004, 8720)}
W8A32_ROUTES = [
    (201, 2071, 1346, _tile(32, 64, 3)), (527, 1156, 1895, _tile(32, 128, 3)), (168, 84, 4949, _tile(64, 64, 3)), (305, 70, 3790, _tile(64, 128, 3)),
    (539, 77, 3716, _tile(32, 128, 2)), (52, 70, 38752, _tile(64, 256, 2)), (162, 81, 39168, _tile(64, 256, 2)), (289, 216, 2022, _tile(64, 64, 3)),
    (45, 834, 20, _rows(3, 1, 8, 2, 1)), (47, 70, 18, _rows(3, 1, 8, 2, 1)), (43, 390, 2670, _rows(6, 2, 4, 2, 1)),
    (68, 71, 34073, _tile(32, 128, 2)), (248, 67, 11625, _tile(128, 128, 2)), (36, 2199, 1583, _rows(3, 2, 4, 3, 1)),
]
