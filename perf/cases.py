"""What a program built on this framework has it do, as cases that can be timed: W8A8 and block-quantised linears, the
quantised products of a decoder layer, whole decoder blocks, mixture-of-experts FFNs in two formats, and
Huffman-coded key/value caches, over the sizes from one token of a small model to a long prompt of a large one.

`listed()` names one case of each kind of work, `draw(rng)` makes further ones of the same ranges, `prepare(case, seed)`
makes the inputs and loads the weights, `run(state)` is one pass through the public entry points (the C ABI's
device-pointer functions where a serving loop would call them, the host-array functions where those are what is called),
`work(case)` is what the pass cannot do without and `tolerance(case)` how far a correct result may be from another.
"""
import ctypes as C
import math

import torch

from peregrine_amd import _ffi, default_context, gguf, huffman, llama, mxfp4, quant

LIB, CHECK = _ffi.lib, _ffi.check
Q4_0, Q4_1, Q8_0 = gguf.Q4_0, gguf.Q4_1, gguf.Q8_0
TYPES = {"q4_0": Q4_0, "q4_1": Q4_1, "q8_0": Q8_0}
BLOCK_BYTES = {"q4_0": 18, "q4_1": 20, "q8_0": 34}


# ---------------------------------------------------------------------------------------------------- inputs
def _ptr(t):
    return C.c_void_p(t.data_ptr())


class _Handle:
    """A library object together with the call that frees it."""

    def __init__(self, free):
        self.h, self._free = C.c_void_p(), free

    def __del__(self):
        if self.h:
            self._free(self.h)
            self.h = C.c_void_p()


class _Rng:
    """Normal and uniform tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def rows(self, m, k):
        """Activations: N(0, 1) with 1 % of the channels twenty times larger, as hidden states have them."""
        a = self.normal(m, k)
        a[:, torch.randperm(k, generator=self.g, device="cuda")[: max(1, k // 100)]] *= 20.0
        return a.contiguous()


def _pack(w, kind):
    """[n, k] f32 on the GPU -> the raw blocks of a GGUF tensor of that type, on the host."""
    b = w.reshape(-1, 32)
    if kind == "q8_0":
        d = (b.abs().amax(1) / 127.0).half()
        q = torch.round(b / d.float().clamp_min(1e-8)[:, None]).clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        parts = (d.view(torch.uint8).reshape(-1, 2), q)
    else:
        if kind == "q4_0":
            top = b.gather(1, b.abs().argmax(1, keepdim=True)).squeeze(1)
            d = (top / -8.0).half()
            df = d.float()
            q = torch.floor(b / torch.where(df == 0, torch.ones_like(df), df)[:, None] + 8.5).clamp_(0, 15).to(torch.uint8)
            head = (d.view(torch.uint8).reshape(-1, 2),)
        else:
            lo = b.amin(1)
            d, m = ((b.amax(1) - lo) / 15.0).half(), lo.half()
            q = torch.round((b - m.float()[:, None]) / d.float().clamp_min(1e-8)[:, None]).clamp_(0, 15).to(torch.uint8)
            head = (d.view(torch.uint8).reshape(-1, 2), m.view(torch.uint8).reshape(-1, 2))
        parts = head + (q[:, 0::2] | (q[:, 1::2] << 4),)
    return torch.cat(parts, 1).cpu().numpy().reshape(-1)


def _gguf(rng, kind, n, k, rows):
    """A weight of N(0, 0.02) kept quantised on the GPU and made ready for products over `rows` rows."""
    return gguf.GgufWeight(_pack(rng.normal(n, k, std=0.02), kind), TYPES[kind], n, k).prepare(rows)


def _qtensor(rng, k, n):
    """An int8 weight of N(0, 0.02) [k, n] on the GPU."""
    w = rng.normal(k, n, std=0.02)
    ctx = default_context()
    torch.cuda.synchronize()
    t = _Handle(lambda h: LIB.pg_qtensor_free(ctx.handle, h))
    CHECK(LIB.pg_qtensor_from_f32_dev(ctx.handle, _ptr(w), k, n, C.byref(t.h)))
    ctx.sync()
    return t


def _mxfp4(w):
    """[n, k] f32 on the GPU -> (codes, block scales) of an MXFP4 tensor, on the host: two FP4 (E2M1) codes a byte, a
    power of two per 32 values that brings the largest of them to 4 .. 8 (what is over 6 becomes 6)."""
    b = w.reshape(-1, 32)
    e = torch.floor(torch.log2(b.abs().amax(1).clamp_min(1e-20))) - 2
    x = b * torch.exp2(-e)[:, None]
    at = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=w.device)
    code = torch.bucketize(x.abs(), at).to(torch.uint8) | ((x < 0).to(torch.uint8) << 3)
    return (code[:, 0::2] | (code[:, 1::2] << 4)).cpu().numpy().reshape(-1), (e + 127).to(torch.uint8).cpu().numpy()


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# ------------------------------------------------------------------------------------------- the kinds of work
class Linear:
    """One linear over an int8 weight, activations and result on the GPU: C[m, n] = A[m, k] . W[k, n]. `w8a8` quantises the
    rows to int8 on the way (quant::matmul_quantized), `w8a32` keeps them in f32 (the numerics of the reference's own GPU
    path, quant::matmul_quantized_gpu)."""

    def draw(rng):
        return {"semantics": rng.choice(["w8a8", "w8a8", "w8a32"]), "m": _log(rng, 2, 2048), "k": _log(rng, 256, 8192), "n": _log(rng, 256, 8192)}

    def prepare(c, seed):
        rng = _Rng(seed)
        w = _qtensor(rng, c["k"], c["n"])
        a, out = rng.rows(c["m"], c["k"]), torch.empty(c["m"], c["n"], device="cuda")
        h = default_context().handle
        if c["semantics"] == "w8a8":
            call = (LIB.pg_matmul_quantized_dev, (h, _ptr(a), c["m"], c["k"], w.h, _ptr(out), None))
        else:
            call = (LIB.pg_matmul_dequant_i8_dev, (h, _ptr(a), c["m"], c["k"], w.h, _ptr(out)))
        return {"calls": [call], "outs": out, "keep": (w, a)}

    def run(s):
        for fn, args in s["calls"]:
            CHECK(fn(*args))
        return s["outs"]

    def work(c):
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": k * n + 4 * n + 4 * m * (k + n), "flops": 2 * m * k * n}

    def tolerance(c):
        return "exact" if c["semantics"] == "w8a8" else {"rel": 1e-5}


class Layer:
    """The seven W8A8 products of one decoder layer over m tokens, as a program runs them: q|k|v and gate|up as products
    over one input, then the output and the down projection. One token is decode, a few tens a batch of users being
    decoded together, thousands a prompt."""

    def draw(rng):
        d = 32 * _log(rng, 16, 128)
        return {"m": _log(rng, 1, 2048), "d": d, "kv": d // rng.choice([2, 4, 8]), "ffn": 8 * int(d * rng.uniform(2.5, 3.5) / 8)}

    def prepare(c, seed):
        rng, h = _Rng(seed), default_context().handle
        m, d, kv, ffn = c["m"], c["d"], c["kv"], c["ffn"]
        w = [_qtensor(rng, k, n) for k, n in ((d, d), (d, kv), (d, kv), (d, d), (d, ffn), (d, ffn), (ffn, d))]
        x, att, act = rng.rows(m, d), rng.rows(m, d), rng.rows(m, ffn)
        outs = [torch.empty(m, n, device="cuda") for n in (d, kv, kv, d, ffn, ffn, d)]

        def table(of):
            return (C.c_void_p * len(of))(*of)

        calls = [
            (LIB.pg_matmul_quantized_multi_dev, (h, _ptr(x), m, d, table([t.h.value for t in w[:3]]), 3, table([o.data_ptr() for o in outs[:3]]))),
            (LIB.pg_matmul_quantized_dev, (h, _ptr(att), m, d, w[3].h, _ptr(outs[3]), None)),
            (LIB.pg_matmul_quantized_multi_dev, (h, _ptr(x), m, d, table([t.h.value for t in w[4:6]]), 2, table([o.data_ptr() for o in outs[4:6]]))),
            (LIB.pg_matmul_quantized_dev, (h, _ptr(act), m, ffn, w[6].h, _ptr(outs[6]), None)),
        ]
        return {"calls": calls, "outs": outs, "keep": (w, x, att, act)}

    run = Linear.run

    def work(c):
        m, d, kv, ffn = c["m"], c["d"], c["kv"], c["ffn"]
        weights = 2 * d * (d + kv) + 3 * d * ffn
        cols = 3 * d + 2 * kv + 2 * ffn
        return {"bytes": weights + 4 * cols + 4 * m * (2 * d + ffn + cols), "flops": 2 * m * weights}

    def tolerance(c):
        return "exact"


class HostLinear:
    """quant::matmul_quantized as the reference's callers have it: activations and result are host arrays, the weight is
    resident."""

    def draw(rng):
        return {"m": _log(rng, 1, 512), "k": _log(rng, 128, 4096), "n": _log(rng, 128, 4096)}

    def prepare(c, seed):
        rng = _Rng(seed)
        qt = quant.quantize_weights(rng.normal(c["k"], c["n"], std=0.02).cpu().numpy(), c["k"], c["n"]).to_gpu()
        return {"a": rng.rows(c["m"], c["k"]).cpu().numpy(), "qt": qt, "m": c["m"], "k": c["k"]}

    def run(s):
        return quant.matmul_quantized(s["a"], s["m"], s["k"], s["qt"])

    def work(c):
        return Linear.work(c)

    def tolerance(c):
        return "exact"


class BlockLinear:
    """One linear over a GGUF tensor that stays in its block format, activations and result on the GPU."""

    def draw(rng):
        return {"type": rng.choice(["q4_0", "q8_0", "q4_1"]), "m": _log(rng, 1, 1024), "k": 32 * _log(rng, 8, 448), "n": _log(rng, 256, 14336)}

    def prepare(c, seed):
        rng = _Rng(seed)
        w = _gguf(rng, c["type"], c["n"], c["k"], c["m"])
        x, out = rng.rows(c["m"], c["k"]), torch.empty(c["m"], c["n"], device="cuda")
        return {"calls": [(LIB.pg_gguf_matmul_dev, (default_context().handle, _ptr(x), c["m"], w._h, _ptr(out)))], "outs": out, "keep": (w, x)}

    run = Linear.run

    def work(c):
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": n * k // 32 * BLOCK_BYTES[c["type"]] + 4 * m * (k + n), "flops": 2 * m * k * n}

    def tolerance(c):
        return {"rel": 5e-5}


class Block:
    """LlamaBlock::forward over projections kept in their block format: `seq` new tokens behind `pos` positions that the
    cache holds. One token is decode, a few are drafted tokens being verified, hundreds a prompt or the next piece of one.
    The cache is taken back to `pos` first, as a program does that drops drafted tokens."""

    def draw(rng):
        d, heads, kv, hd, ffn = rng.choice([(1024, 16, 4, 64, 2816), (2048, 32, 8, 64, 8192), (2048, 16, 2, 128, 5632), (4096, 32, 8, 128, 14336)])
        seq = _log(rng, 1, 1024)
        return {"type": rng.choice(["q4_0", "q8_0"]), "seq": seq, "pos": _log(rng, 1, 8192) if seq < 128 else rng.choice([0, _log(rng, 64, 2048)]),
                "d": d, "heads": heads, "kv_heads": kv, "head_dim": hd, "ffn": ffn}

    def _shapes(c):
        d, q, kv, f = c["d"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["ffn"]
        return ((q, d), (kv, d), (kv, d), (d, q), (f, d), (f, d), (d, f))

    def prepare(c, seed):
        rng, ctx = _Rng(seed), default_context()
        seq, pos, d, kv, hd = c["seq"], c["pos"], c["d"], c["kv_heads"], c["head_dim"]
        ws = [_gguf(rng, c["type"], n, k, seq) for n, k in Block._shapes(c)]
        block = llama.LlamaBlock(d, c["heads"], kv, hd, c["ffn"], pos + seq, 500000.0, 1e-5)
        norms = 1.0 + rng.normal(2, d, std=0.1).cpu().numpy()
        block.set_weights(*ws, norms[0], norms[1])
        cache = block.new_cache()
        k, v = rng.normal(kv, pos + seq, hd), rng.normal(kv, pos + seq, hd, std=0.3)
        torch.cuda.synchronize()
        CHECK(LIB.pg_kv_cache_append_dev(ctx.handle, cache._h, _ptr(k), _ptr(v), pos + seq))
        ctx.sync()
        h, out = rng.rows(seq, d), torch.empty(seq, d, device="cuda")
        calls = [(LIB.pg_kv_cache_rollback_to, (cache._h, pos)), (LIB.pg_llama_block_forward_dev, (ctx.handle, block._h, _ptr(h), seq, cache._h, _ptr(out)))]
        return {"calls": calls, "outs": out, "keep": (ws, block, cache, h)}

    run = Linear.run

    def work(c):
        seq, pos = c["seq"], c["pos"]
        weights = sum(n * k for n, k in Block._shapes(c))
        q, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        return {"bytes": weights // 32 * BLOCK_BYTES[c["type"]] + 8 * kv * (pos + seq) + 8 * kv * seq + 8 * seq * c["d"],
                "flops": 2 * seq * weights + 4 * q * (seq * pos + seq * (seq + 1) // 2)}

    def tolerance(c):
        return {"rel": 1e-4}


class Experts:
    """MoELayer::forward after its router's product, over block-quantised experts: softmax, the top_k experts of each token,
    gated FFN, weighted sum. Few tokens touch few experts, a batch all of them."""

    def draw(rng):
        E = rng.choice([4, 8, 16])
        return {"type": rng.choice(["q8_0", "q8_0", "q4_0"]), "tokens": _log(rng, 1, 256), "d": 32 * _log(rng, 16, 96), "ffn": 32 * _log(rng, 32, 2048 // E),
                "experts": E, "top_k": rng.choice([1, 2, 2, 4]), "act": rng.choice(["silu", "gelu"])}

    def prepare(c, seed):
        rng, h = _Rng(seed), default_context().handle
        T, d, ffn, E = c["tokens"], c["d"], c["ffn"], c["experts"]
        ws = [[_gguf(rng, c["type"], n, k, T) for _ in range(E)] for n, k in ((ffn, d), (ffn, d), (d, ffn))]
        tabs = [(C.c_void_p * E)(*[w._h.value for w in of]) for of in ws]
        x, logits, out = rng.rows(T, d), rng.normal(T, E), torch.empty(T, d, device="cuda")
        act = _ffi.ACT_SILU if c["act"] == "silu" else _ffi.ACT_GELU_TANH
        call = (LIB.pg_moe_ffn_dev, (h, _ptr(x), T, _ptr(logits), E, c["top_k"], *tabs, act, _ptr(out)))
        return {"calls": [call], "outs": out, "keep": (ws, x, logits)}

    run = Linear.run

    def work(c):
        T, d, ffn, E, k = c["tokens"], c["d"], c["ffn"], c["experts"], c["top_k"]
        hit = E * (1 - (1 - k / E) ** T)  # experts that T tokens are expected to choose between them
        return {"bytes": hit * 3 * d * ffn // 32 * BLOCK_BYTES[c["type"]] + 8 * T * d + 4 * T * E, "flops": 6 * T * k * d * ffn}

    def tolerance(c):
        return {"rel": 1e-4}


class Mxfp4Experts:
    """The same layer over MXFP4 experts with biases and the clamped, interleaved SwiGLU, routed by the caller (top-k of the
    logits, softmax over the k)."""

    def draw(rng):
        return {"tokens": _log(rng, 1, 512), "hidden": 32 * _log(rng, 16, 90), "inter": 32 * _log(rng, 16, 90), "experts": rng.choice([8, 16, 32]), "top_k": rng.choice([2, 4])}

    def prepare(c, seed):
        rng = _Rng(seed)
        T, hid, inter, E, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top_k"]
        ex = []
        for _ in range(E):
            b1, s1 = _mxfp4(rng.normal(2 * inter, hid, std=0.02))
            b2, s2 = _mxfp4(rng.normal(hid, inter, std=0.02))
            bias = rng.normal(2 * inter + hid, std=0.1).cpu().numpy()
            ex.append(mxfp4.Mxfp4Expert(hid, inter, 1.702, 7.0, b1, s1, b2, s2, bias[: 2 * inter], bias[2 * inter:]))
        x, top = rng.rows(T, hid), torch.topk(rng.normal(T, E), k, dim=1)
        idx, wt = top.indices.to(torch.int32).contiguous(), torch.softmax(top.values, 1).contiguous()
        out = torch.empty(T, hid, device="cuda")
        tab = C.cast((C.c_void_p * E)(*[e._h.value for e in ex]), C.POINTER(C.c_void_p))
        call = (LIB.pg_mxfp4_moe_ffn_routed_dev, (default_context().handle, _ptr(x), T, _ptr(idx), _ptr(wt), k, tab, E, _ptr(out)))
        return {"calls": [call], "outs": out, "keep": (ex, x, idx, wt, tab)}

    run = Linear.run

    def work(c):
        T, hid, inter, E, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top_k"]
        hit = E * (1 - (1 - k / E) ** T)
        return {"bytes": hit * (3 * hid * inter // 32 * 17 + 4 * (2 * inter + hid)) + 8 * T * hid + 8 * T * k, "flops": 6 * T * k * hid * inter}

    def tolerance(c):
        return {"rel": 1e-4}


class HuffmanCache:
    """A sequence under a Huffman-coded key/value cache, from its first token to its end: `tokens` positions come in `piece`
    at a time, what leaves the window is coded in chunks, and the keys and values are read back for attention."""

    def draw(rng):
        tokens, chunk = _log(rng, 200, 3000), rng.choice([64, 128, 256])
        return {"tokens": tokens, "piece": max(tokens // 12, _log(rng, 32, 1024)), "chunk": chunk, "window": chunk * rng.choice([1, 2]),
                "heads": rng.choice([2, 4, 8]), "head_dim": rng.choice([64, 128])}

    def prepare(c, seed):
        rng = _Rng(seed)
        T, heads, hd = c["tokens"], c["heads"], c["head_dim"]
        sizes = [min(c["piece"], T - at) for at in range(0, T, c["piece"])]
        pieces = [(rng.normal(heads, n, hd), rng.normal(heads, n, hd, std=0.3), n) for n in sizes]
        return {"pieces": pieces, "args": (heads, hd, c["window"], c["chunk"]), "outs": [torch.empty(heads, T, hd, device="cuda") for _ in range(2)]}

    def run(s):
        cache = huffman.HuffmanKVCache(*s["args"])
        h = cache.ctx.handle
        for k, v, n in s["pieces"]:
            CHECK(LIB.pg_huffman_kv_cache_append_dev(h, cache._h, _ptr(k), _ptr(v), n))
        k, v = s["outs"]
        CHECK(LIB.pg_huffman_kv_cache_get_kv_dev(h, cache._h, _ptr(k), _ptr(v)))
        cache.free()
        return s["outs"]

    def work(c):
        n = 2 * c["tokens"] * c["heads"] * c["head_dim"]
        return {"bytes": 8 * n + 2 * 0.9 * n, "flops": 2 * n}  # values in and out in f32, and about 7.1 bits of code each, written and read

    def tolerance(c):
        return "exact"


KINDS = {"linear": Linear, "layer": Layer, "host_linear": HostLinear, "block_linear": BlockLinear, "block": Block, "experts": Experts,
         "mxfp4_experts": Mxfp4Experts, "huffman_cache": HuffmanCache}


def listed():
    wide = {"d": 4096, "heads": 32, "kv_heads": 8, "head_dim": 128, "ffn": 14336}
    return [
        # the smallest call: three tokens through one projection of a small model
        {"name": "linear_w8a8_3x768x3072", "kind": "linear", "semantics": "w8a8", "m": 3, "k": 768, "n": 3072},
        # f32 activations over an int8 weight, a ragged number of rows
        {"name": "linear_w8a32_197x1024x4096", "kind": "linear", "semantics": "w8a32", "m": 197, "k": 1024, "n": 4096},
        # int8 decode: one token through a layer of the benchmark's size, and a ragged batch of users through a smaller one
        {"name": "layer_w8a8_1", "kind": "layer", "m": 1, "d": 4096, "kv": 1024, "ffn": 14336},
        {"name": "layer_w8a8_27_ragged", "kind": "layer", "m": 27, "d": 2016, "kv": 504, "ffn": 5432},
        # int8 prefill: the benchmark's headline, a prompt of 2048 tokens
        {"name": "layer_w8a8_2048", "kind": "layer", "m": 2048, "d": 4096, "kv": 1024, "ffn": 14336},
        # the reference's own int8 benchmark, host arrays in and out
        {"name": "host_w8a8_196x768x3072", "kind": "host_linear", "m": 196, "k": 768, "n": 3072},
        # a file's less common 4-bit format, a dozen users
        {"name": "gguf_q4_1_12x4096x4096", "kind": "block_linear", "type": "q4_1", "m": 12, "k": 4096, "n": 4096},
        # a 4-bit model decoding one token of a long conversation, and an 8-bit one reading the next piece of a prompt
        {"name": "block_q4_0_decode_at_4095", "kind": "block", "type": "q4_0", "seq": 1, "pos": 4095, **wide},
        {"name": "block_q8_0_prefill_777", "kind": "block", "type": "q8_0", "seq": 777, "pos": 100, **wide},
        # experts: a decoding batch over 8-bit ones (half the width of the benchmark's), and a smaller one over MXFP4 ones
        {"name": "experts_q8_0_64_tokens", "kind": "experts", "type": "q8_0", "tokens": 64, "d": 3072, "ffn": 8192, "experts": 8, "top_k": 2, "act": "silu"},
        {"name": "experts_mxfp4_20_tokens", "kind": "mxfp4_experts", "tokens": 20, "hidden": 2880, "inter": 2880, "experts": 32, "top_k": 4},
        # coded keys and values: a prompt in pieces of 512 and its read-back (encode and decode)
        {"name": "huffman_cache_3000_tokens", "kind": "huffman_cache", "tokens": 3000, "piece": 512, "chunk": 256, "window": 512, "heads": 8, "head_dim": 128},
    ]


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(list(KINDS))
        c = {"kind": kind, **KINDS[kind].draw(rng)}
        if _cost(c) <= most:
            return c


def _cost(c):
    """Of the order of the time a pass takes, for the choice of drawn cases."""
    w = work(c)
    return max(w["bytes"], w["flops"] / 400)


def prepare(case, seed):
    s = KINDS[case["kind"]].prepare(case, seed)
    s["kind"] = KINDS[case["kind"]]
    torch.cuda.synchronize()
    return s


def run(state):
    return state["kind"].run(state)


def work(case):
    return KINDS[case["kind"]].work(case)


def tolerance(case):
    return KINDS[case["kind"]].tolerance(case)
