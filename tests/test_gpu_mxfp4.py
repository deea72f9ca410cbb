"""GPU parity of the MXFP4 path (examples/gpt_oss/moe.rs) against the CPU oracle, through the
C ABI.  Bar: the block-dequant contract, 1e-3 relative (H.assert_close_rel); the fixed-point
kernel is exact up to the final f32 roundings, so the tests also hold it to 2e-5."""
import ctypes as C
import sys

import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu
RTOL_CONTRACT, RTOL_ACHIEVED = 1e-3, 2e-5


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _weights(rng, n, k, lo=118, hi=124):
    return (rng.integers(0, 256, n * k // 2, dtype=np.uint8), rng.integers(lo, hi, n * k // 32, dtype=np.uint8))


def test_mxfp4_codes_scales_and_order_exact(ctx, orc):
    """One-hot inputs read single weights back: every code, both nibbles, a spread of scale bytes."""
    from peregrine_amd import mxfp4
    in_dim, out_dim = 64, 16
    blocks = np.zeros((out_dim, 2, 16), np.uint8)
    for r in range(out_dim):
        blocks[r, 0, 0] = r                    # code r in the low nibble of element 0
        blocks[r, 1, 5] = r << 4               # code r in the high nibble of element 32 + 11
    scales = np.full((out_dim, 2), 127, np.uint8)
    for pos in (0, 1, 43, 42):
        x = np.zeros(in_dim, np.float32)
        x[pos] = 3.0
        got = mxfp4.mxfp4_matmul(x, blocks, scales, out_dim, in_dim, ctx)
        assert (got == orc.mxfp4_matmul(x, blocks, scales, out_dim, in_dim)).all(), pos
    x = np.zeros(in_dim, np.float32)
    x[0] = 1.0
    one = np.zeros((1, 2, 16), np.uint8)
    one[0, 0, 0] = 2
    for e in (0, 1, 2, 60, 126, 127, 128, 200, 253, 254):
        s = np.array([[e, 127]], np.uint8)
        got = mxfp4.mxfp4_matmul(x, one, s, 1, in_dim, ctx)[0]
        want = orc.mxfp4_matmul(x, one, s, 1, in_dim)[0]
        assert got == want, (e, got, want)


@pytest.mark.parametrize("out_dim,in_dim", [(5760, 2880), (2880, 2880), (33, 96), (1, 32), (257, 8192 + 32)])
def test_mxfp4_matmul(ctx, orc, out_dim, in_dim):
    """gpt-oss shapes (hidden 2880, mlp1 rows 2 x 2880) and ragged ones."""
    from peregrine_amd import mxfp4
    say(f"mxfp4 matmul [{in_dim}] -> [{out_dim}]")
    rng = np.random.default_rng(out_dim + in_dim)
    b, s = _weights(rng, out_dim, in_dim)
    x = orc.rng_normal(out_dim, in_dim)
    x[::97] *= 20.0
    got = mxfp4.mxfp4_matmul(x, b, s, out_dim, in_dim, ctx)
    want = orc.mxfp4_matmul(x, b, s, out_dim, in_dim)
    H.assert_close_rel(got, want, RTOL_CONTRACT, "mxfp4 contract")
    H.assert_close_rel(got, want, RTOL_ACHIEVED, "mxfp4 achieved")


def test_mxfp4_resident_weight_rows_and_errors(ctx, orc):
    from peregrine_amd import mxfp4, _ffi
    rng = np.random.default_rng(5)
    out_dim, in_dim, m = 200, 256, 7
    b, s = _weights(rng, out_dim, in_dim, 100, 150)
    w = mxfp4.upload(b, s, out_dim, in_dim, ctx)
    assert (w.n_out, w.k_in, w.ggml_type) == (out_dim, in_dim, _ffi.MXFP4)
    x = orc.rng_normal(3, m * in_dim).reshape(m, in_dim)
    got = w.matmul(x, m).reshape(m, out_dim)
    for i in range(m):
        H.assert_close_rel(got[i], orc.mxfp4_matmul(x[i], b, s, out_dim, in_dim), RTOL_ACHIEVED, f"row {i}")
    with pytest.raises(ValueError):
        mxfp4.mxfp4_matmul(x[0], b, s, out_dim, in_dim + 1, ctx)
    with pytest.raises(ValueError):
        mxfp4.mxfp4_matmul(x[0], b[:-1], s, out_dim, in_dim, ctx)


@pytest.mark.parametrize("m", [1, 3, 40])
def test_mxfp4_expert_forward(ctx, orc, m):
    from peregrine_amd import mxfp4
    hidden, inter, alpha, clamp = 2880, 2880, 1.702, 7.0
    say(f"mxfp4 expert hidden={hidden} intermediate={inter} m={m}")
    rng = np.random.default_rng(21)
    b1, s1 = _weights(rng, 2 * inter, hidden, 116, 120)
    b2, s2 = _weights(rng, hidden, inter, 116, 120)
    bias1 = orc.rng_normal(1, 2 * inter)
    bias2 = orc.rng_normal(2, hidden)
    ex = mxfp4.Mxfp4Expert(hidden, inter, alpha, clamp, b1, s1, b2, s2, bias1, bias2, ctx)
    x = orc.rng_normal(4, m * hidden).reshape(m, hidden)
    got = ex.forward(x if m > 1 else x[0]).reshape(m, hidden)
    for i in range(0, m, 1 if m < 8 else 9):   # (24 rows and more: both products take the matrix-core block product)
        want = orc.mxfp4_expert_forward(x[i], hidden, inter, alpha, clamp, b1, s1, b2, s2, bias1, bias2)
        H.assert_close_rel(got[i], want, RTOL_CONTRACT, f"mxfp4 expert row {i}")
        H.assert_close_rel(got[i], want, 1e-4 if m < 8 else 6e-4, f"mxfp4 expert row {i} (achieved)")


@pytest.mark.parametrize("out_dim,in_dim,m", [(4096, 14336, 1), (14336, 4096, 2), (600, 512, 5), (48, 28160, 1), (8200, 1024, 3)])
def test_mxfp4_workgroup_shapes(ctx, orc, out_dim, in_dim, m):
    """One case per launch shape of the product kernel: 16 wavefronts on one row group (few row groups),
    8 wavefronts on 1, 2 or 4 row groups, one to three activation rows per pass, several passes (m = 5),
    and K at the upper limit of what the digit planes in LDS hold."""
    from peregrine_amd import mxfp4
    say(f"mxfp4 shapes [{m} x {in_dim}] -> [{out_dim}]")
    rng = np.random.default_rng(out_dim * 7 + in_dim + m)
    b, s = _weights(rng, out_dim, in_dim)
    w = mxfp4.upload(b, s, out_dim, in_dim, ctx)
    x = orc.rng_normal(m + 11, m * in_dim).reshape(m, in_dim)
    x[:, ::89] *= 30.0
    got = w.matmul(x, m).reshape(m, out_dim)
    rows = rng.choice(out_dim, size=min(out_dim, 256), replace=False)   # the oracle on a sample of the weight rows
    bb = b.reshape(out_dim, -1)[rows].reshape(-1)
    ss = s.reshape(out_dim, -1)[rows].reshape(-1)
    for i in range(m):
        want = orc.mxfp4_matmul(x[i], bb, ss, len(rows), in_dim)
        H.assert_close_rel(got[i][rows], want, RTOL_ACHIEVED, f"row {i}")
    w.free()


RTOL_TILES = 1e-4   # four planes of base-32 digits per activation block: 20 bits under the block's largest value


@pytest.mark.parametrize("out_dim,in_dim,m,lo,hi,plan", [
    (2880, 2880, 24, 118, 124, (1, 2, 3)), (8192, 4096, 16, 118, 124, (1, 1, 4)), (5760, 2880, 100, 118, 124, (1, 4, 2)),
    (600, 4096, 300, 104, 144, (1, 4, 4)), (520, 512, 40, 100, 150, (1, 4, 1)),          # narrow row tiles, K in runs
    (8192, 256, 512, 100, 150, (2, 4, 1)), (14336, 128, 640, 110, 140, (4, 4, 1)),          # wider row tiles, one run
    (70000, 512, 16, 110, 140, (2, 1, 1)), (70000, 512, 32, 110, 140, (2, 2, 1)),
    (140000, 256, 16, 110, 140, (4, 1, 1)), (140000, 256, 30, 110, 140, (4, 2, 1)),
    (37, 96, 50, 0, 255, (1, 4, 1)),                                                         # every scale byte, ragged everything
])
def test_mxfp4_many_rows(ctx, orc, out_dim, in_dim, m, lo, hi, plan):
    """From 16 activation rows on (24 for a small tensor) the tile kernel on the scaled matrix-core instruction takes the
    product, whatever the block scales: the rows as four planes of base-32 digits (RTOL_TILES with x25 outlier
    channels).  plan = (groups of 16 weight rows per wavefront, groups of 16 tokens per workgroup, runs of K) the
    launcher picks on a 256-CU part.  One row on the same tensor afterwards still takes the decode kernel."""
    from peregrine_amd import mxfp4, _ffi
    say(f"mxfp4 many rows [{m} x {in_dim}] -> [{out_dim}] scales {lo}..{hi - 1}")
    v, got_plan = [C.c_size_t() for _ in range(6)], [C.c_int() for _ in range(3)]
    _ffi.check(_ffi.lib.pg_audit_mxfp4_tiles(256, out_dim, in_dim, m, *[C.byref(x) for x in v], *[C.byref(x) for x in got_plan]))   # an MI355X has 256 CUs
    assert tuple(x.value for x in got_plan) == plan
    rng = np.random.default_rng(out_dim + 3 * in_dim + m)
    b, s = _weights(rng, out_dim, in_dim, lo, hi)
    if hi - lo < 200:
        s[:4] = (lo, hi - 1, 0, lo)            # both ends of the range and a zero block in row 0
    else:
        s[s == 255] = 254                      # (255 is NaN: its own test below)
    w = mxfp4.upload(b, s, out_dim, in_dim, ctx)
    x = orc.rng_normal(m + 5, m * in_dim).reshape(m, in_dim)
    x[:, ::61] *= 25.0
    ctx.profile_begin()
    got = w.matmul(x, m).reshape(m, out_dim)
    prof = ctx.profile_end()
    assert "mxfp4_tiles" in prof and "mxfp4_planes" in prof and ("gguf_mm_sum_parts" in prof) == (got_plan[2].value > 1), prof
    rows = np.concatenate([[0, out_dim - 1], rng.choice(np.arange(1, out_dim), size=min(out_dim - 1, 94), replace=False)])
    bb = b.reshape(out_dim, -1)[rows].reshape(-1)
    ss = s.reshape(out_dim, -1)[rows].reshape(-1)
    wide = hi - lo >= 200                       # scales spread over 2^254: compare where the f32 reference itself is finite
    for i in list(range(0, m, max(1, m // 12))) + [m - 1]:
        want = orc.mxfp4_matmul(x[i], bb, ss, len(rows), in_dim)
        ok = np.isfinite(want) & (np.abs(want) < 1e30) if wide else np.ones(len(rows), bool)
        assert ok.any()
        if wide:                                # each output has its own magnitude: element by element, relative to itself
            rel = np.abs(got[i][rows][ok].astype(np.float64) - want[ok]) / np.maximum(np.abs(want[ok].astype(np.float64)), 1e-300)
            assert np.median(rel) <= RTOL_TILES and (rel <= 5e-2).all(), (i, np.median(rel), rel.max())
        else:
            H.assert_close_rel(got[i][rows], want, RTOL_CONTRACT, f"row {i} (contract)")
            H.assert_close_rel(got[i][rows], want, RTOL_TILES, f"row {i} (achieved)")
    one = w.matmul(x[3], 1)
    if not wide:
        H.assert_close_rel(one[rows], orc.mxfp4_matmul(x[3], bb, ss, len(rows), in_dim), RTOL_ACHIEVED, "one row afterwards")
    xb = x.copy()
    xb[2, 7] = np.nan                           # a NaN poisons its row and no other
    gotb = w.matmul(xb, m).reshape(m, out_dim)
    assert np.isnan(gotb[2]).all() and (gotb[[0, 1, 3, m - 1]] == got[[0, 1, 3, m - 1]]).all()
    w.free()


def test_mxfp4_limits_and_non_finite(ctx, orc):
    from peregrine_amd import mxfp4, _ffi
    rng = np.random.default_rng(9)
    b, s = _weights(rng, 16, 28672)
    with pytest.raises(_ffi.PeregrineError):   # the row's digit planes no longer fit in LDS
        mxfp4.mxfp4_matmul(np.zeros(28672, np.float32), b, s, 16, 28672, ctx)
    out_dim, in_dim = 40, 128
    b, s = _weights(rng, out_dim, in_dim)
    x = orc.rng_normal(1, in_dim)
    base = mxfp4.mxfp4_matmul(x, b, s, out_dim, in_dim, ctx)
    assert np.isfinite(base).all()
    for bad in (np.nan, np.inf, -np.inf):       # the reference's f32 sum turns inf or NaN in every row as well
        xb = x.copy()
        xb[37] = bad
        got = mxfp4.mxfp4_matmul(xb, b, s, out_dim, in_dim, ctx)
        want = orc.mxfp4_matmul(xb, b, s, out_dim, in_dim)
        assert not np.isfinite(got).any() and not np.isfinite(want).any()
    s2 = s.copy().reshape(out_dim, -1)
    s2[3, 1] = 255                              # f32::from_bits(255 << 23) = inf: that row is lost, the others are not
    got = mxfp4.mxfp4_matmul(x, b, s2.reshape(-1), out_dim, in_dim, ctx)
    assert not np.isfinite(got[3]) and not np.isfinite(orc.mxfp4_matmul(x, b, s2.reshape(-1), out_dim, in_dim)[3])
    keep = np.arange(out_dim) != 3
    assert (got[keep] == base[keep]).all()
    s3 = s.copy().reshape(out_dim, -1)
    s3[5, :] = 0                                # f32::from_bits(0) = 0.0: the row is exactly zero
    got = mxfp4.mxfp4_matmul(x, b, s3.reshape(-1), out_dim, in_dim, ctx)
    assert got[5] == 0.0 and orc.mxfp4_matmul(x, b, s3.reshape(-1), out_dim, in_dim)[5] == 0.0


@pytest.mark.parametrize("hidden,inter,E,top_k,T", [
    (64, 96, 4, 2, 1), (128, 64, 32, 4, 8), (2880, 2880, 8, 4, 2),      # few pairs: the decode kernel, a workgroup column per pair
    (64, 96, 5, 3, 7), (256, 160, 8, 2, 64), (512, 512, 8, 4, 300), (128, 64, 32, 4, 40),
    (2880, 2880, 4, 2, 150),        # the gpt-oss expert shape; 75 tokens an expert on average
])
def test_mxfp4_moe_routed_follows_the_oracle(ctx, orc, hidden, inter, E, top_k, T):
    """MoELayer::forward over MXFP4 experts (examples/gpt_oss/moe.rs:286-352), every product one launch over all
    experts, against the reference's per-token walk; experts with no token, with one, and with more than a tile's."""
    from peregrine_amd import mxfp4
    from test_oracle_formats_pins import _mx_expert
    say(f"mxfp4 moe hidden={hidden} inter={inter} E={E} top_k={top_k} T={T}")
    rng = np.random.default_rng(hidden + inter + E + T)
    raw = [_mx_expert(rng, hidden, inter) for _ in range(E)]
    experts = [mxfp4.Mxfp4Expert(hidden, inter, 1.702, 7.0, *r, ctx=ctx) for r in raw]
    x = orc.rng_normal(T + 11, T * hidden).reshape(T, hidden)
    x[:, ::37] *= 10.0
    logits = rng.standard_normal((T, E)).astype(np.float32)
    logits[:, 0] -= 8.0                                    # expert 0 is (almost) never chosen
    idx, w = orc.gpt_oss_route(logits, np.zeros(E, np.float32), T, E, top_k)
    got = mxfp4.moe_forward_routed(x, idx, w, experts, ctx)
    rows = list(range(0, T, max(1, T // 10))) + [T - 1]
    want = orc.mxfp4_moe_routed(x[rows], len(rows), hidden, inter, 1.702, 7.0, top_k, np.asarray(idx).reshape(T, top_k)[rows],
                                np.asarray(w).reshape(T, top_k)[rows], raw)
    for j, t in enumerate(rows):
        H.assert_close_rel(got[t], want[j], RTOL_CONTRACT, f"token {t} (contract)")
        H.assert_close_rel(got[t], want[j], 2e-4, f"token {t} (achieved)")
    # one expert called alone on the tokens routed to it gives the same rows as the grouped launch did for those pairs
    e = int(np.bincount(np.asarray(idx).reshape(-1), minlength=E).argmax())
    toks = [t for t in range(T) if e in np.asarray(idx).reshape(T, top_k)[t]][:5]
    if top_k == 1 and toks:
        alone = experts[e].forward(x[toks])
        H.assert_close_rel(got[toks] / np.asarray(w).reshape(T, top_k)[toks], alone, 2e-4, "one expert alone")
    with pytest.raises(ValueError):
        mxfp4.moe_forward_routed(x, np.asarray(idx).reshape(T, top_k), np.asarray(w).reshape(T, top_k)[:, :1], experts, ctx)
    from peregrine_amd import _ffi
    bad = np.asarray(idx, np.int32).reshape(T, top_k).copy()
    bad[T - 1, 0] = E                                      # the reference's self.experts[expert_idx] would panic
    with pytest.raises(_ffi.PeregrineError):
        mxfp4.moe_forward_routed(x, bad, w, experts, ctx)
    if top_k > 1:
        bad[T - 1, 0] = bad[T - 1, 1]                      # an expert named twice by one token
        with pytest.raises(_ffi.PeregrineError):
            mxfp4.moe_forward_routed(x, bad, w, experts, ctx)
    for ex in experts:
        ex.free()


@pytest.mark.parametrize("hidden,inter", [(96, 64), (1120, 544), (2880, 288), (544, 2112)])
def test_mxfp4_moe_tiles_with_few_slots(ctx, orc, hidden, inter):
    """Experts with 0 to 17 tokens in one launch: up to 4 and up to 8 slots of a token tile go through narrower forms of the
    product (several digit planes of a token in one operand); 17 is a full tile and one slot.  A token that holds a NaN
    leaves the others of its tile as they are.  Bound as for the routed test above: 20 bits under a block's largest value."""
    from peregrine_amd import mxfp4
    from test_oracle_formats_pins import _mx_expert
    say(f"mxfp4 moe, few slots, hidden={hidden} inter={inter}")
    rng = np.random.default_rng(hidden + inter)
    counts = [0, 1, 3, 4, 5, 8, 9, 15, 16, 17, 2]          # 80 pairs over 11 experts: tiles of 16 slots
    E, T = len(counts), sum(counts)
    raw = [_mx_expert(rng, hidden, inter) for _ in range(E)]
    experts = [mxfp4.Mxfp4Expert(hidden, inter, 1.702, 7.0, *r, ctx=ctx) for r in raw]
    idx = rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts)).reshape(T, 1)
    w = rng.uniform(0.2, 1.0, (T, 1)).astype(np.float32)
    x = orc.rng_normal(T + 3, T * hidden).reshape(T, hidden)
    x[:, ::37] *= 10.0
    got = mxfp4.moe_forward_routed(x, idx, w, experts, ctx)
    want = orc.mxfp4_moe_routed(x, T, hidden, inter, 1.702, 7.0, 1, idx, w, raw)
    for t in range(T):
        H.assert_close_rel(got[t], want[t], 2e-4, f"token {t}, one of {counts[idx[t, 0]]} of its expert")
    for n in (3, 8):
        t = int(np.flatnonzero(idx[:, 0] == counts.index(n))[0])
        xn = x.copy()
        xn[t, hidden // 2] = np.nan
        other = mxfp4.moe_forward_routed(xn, idx, w, experts, ctx)
        assert not np.isfinite(other[t]).any()
        keep = np.arange(T) != t
        assert (other[keep] == got[keep]).all()
    for ex in experts:
        ex.free()


@pytest.mark.parametrize("hidden,inter,E,top_k,T,pairs", [
    (512, 512, 8, 2, 32, True), (512, 512, 8, 5, 13, False),         # 64 and 65 pairs
    (512, 512, 8, 3, 21, True), (1024, 1024, 4, 2, 25, True), (1024, 1024, 4, 2, 26, False),   # 63; both sides of the estimates
    (64, 96, 40, 1, 64, True), (64, 96, 33, 5, 13, False),           # up to 64 pairs of more experts than that are always pairs
])
def test_mxfp4_moe_pairs_or_tiles(ctx, orc, hidden, inter, E, top_k, T, pairs):
    """Up to 64 (token, expert) pairs go one by one, also where pairs share experts if the estimates say so; 65 never do.
    Bounds as for the routed test: exact digits one by one, 20 bits under a block's largest value in tiles."""
    from peregrine_amd import mxfp4
    from test_oracle_formats_pins import _mx_expert
    say(f"mxfp4 moe pairs or tiles hidden={hidden} inter={inter} E={E} top_k={top_k} T={T}")
    rng = np.random.default_rng(hidden + E + T)
    raw = [_mx_expert(rng, hidden, inter) for _ in range(E)]
    experts = [mxfp4.Mxfp4Expert(hidden, inter, 1.702, 7.0, *r, ctx=ctx) for r in raw]
    x = orc.rng_normal(T + 5, T * hidden).reshape(T, hidden)
    x[:, ::37] *= 10.0
    idx = np.stack([rng.permutation(E)[:top_k] for _ in range(T)]).astype(np.int32)
    w = rng.uniform(0.2, 1.0, (T, top_k)).astype(np.float32)
    ctx.profile_begin()
    got = mxfp4.moe_forward_routed(x, idx, w, experts, ctx)
    prof = ctx.profile_end()
    assert ("mxfp4_rows_pairs" in prof) == pairs and ("mxfp4_tiles_grouped" in prof) != pairs, sorted(prof)
    want = orc.mxfp4_moe_routed(x, T, hidden, inter, 1.702, 7.0, top_k, idx, w, raw)
    for t in range(T):
        H.assert_close_rel(got[t], want[t], 2e-4, f"token {t}")
    for ex in experts:
        ex.free()


@pytest.mark.parametrize("hidden,inter,E,top_k,T", [
    (544, 2112, 16, 4, 90), (1440, 1440, 4, 4, 130), (1056, 1056, 8, 4, 300),   # 32 slots: 16 to 64 weight rows a wavefront, 4 and 8 of them
    (1120, 544, 8, 4, 40), (352, 96, 2, 2, 70),                                 # 16 slots; few row groups
    (2080, 1056, 16, 4, 700), (544, 1056, 2, 2, 1500),                          # 64 slots
])
def test_mxfp4_moe_tilings(ctx, orc, hidden, inter, E, top_k, T):
    """Every tiling that the estimates choose from, at ragged row groups and last tiles."""
    test_mxfp4_moe_routed_follows_the_oracle(ctx, orc, hidden, inter, E, top_k, T)


@pytest.mark.parametrize("hidden,inter,E,top_k,T", [(96, 480, 130, 4, 194), (96, 992, 130, 4, 194)])
def test_mxfp4_moe_narrow_tilings(ctx, orc, hidden, inter, E, top_k, T):
    """32 and 64 weight rows a wavefront over tiles of 16 slots: six tokens an expert, so full tiles and both narrow forms."""
    test_mxfp4_moe_routed_follows_the_oracle(ctx, orc, hidden, inter, E, top_k, T)


@pytest.mark.parametrize("m", [24, 40, 70])
def test_mxfp4_tiles_digits_at_their_ends(ctx, m):
    """The largest digits of every plane, and the largest scales: one weight of 1 a row, so a product is its block's first value.  A
    block is held in units of 2^-19 of the power of two above its largest value, which the first is: half a unit is at most 2^-19
    of it, and the result is rounded once more (2^-24)."""
    from peregrine_amd import mxfp4
    k, n = 160, 33
    rng = np.random.default_rng(m)
    b = np.zeros((n, k // 2), np.uint8)
    b[:, 0] = 0x02                                         # element 0: 1.0
    s = np.full(n * k // 32, 97, np.uint8)                 # 2^-30
    ends = [3.4028234663852886e38, -3.4028234663852886e38, 1.0, -1.0, 2.0 ** -60, 2.0 ** 20 - 1, 541200.0, -541200.0, 16.0, 17.0, 528.0, -16912.0]
    x = np.zeros((m, k), np.float32)
    x[:, 0] = np.resize(np.array(ends, np.float32), m)
    x[:, 1:32] = x[:, :1] * rng.uniform(-1, 1, (m, 31)).astype(np.float32)
    x[:, 40] = 7.0                                         # (a block without weights)
    w = mxfp4.upload(b.reshape(-1), s, n, k, ctx)
    got = w.matmul(x, m).reshape(m, n).astype(np.float64)
    want = x[:, :1].astype(np.float64) * 2.0 ** -30
    assert (np.abs(got - want) <= np.abs(want) * (2.0 ** -19 + 2.0 ** -24)).all()
    w.free()


@pytest.mark.parametrize("E,T", [(63, 30), (64, 41), (65, 30), (127, 60), (128, 200), (129, 23), (256, 300)])
def test_mxfp4_moe_finds_the_expert_of_a_tile(ctx, orc, E, T):
    """The offsets of 64 experts are looked through at a time: the last expert of a run, the first of the next, and one run more for
    the end of the last tile."""
    test_mxfp4_moe_routed_follows_the_oracle(ctx, orc, 64, 96, E, 3, T)


@pytest.mark.parametrize("E,top_k,T,one", [(32, 4, 373, True), (32, 2, 422, True), (64, 6, 190, True), (64, 4, 512, True), (64, 4, 513, False), (256, 2, 256, True),
                                             (4, 2, 16384, True), (4, 2, 16385, False), (2, 2, 24576, True), (2, 2, 24577, False)])
def test_mxfp4_moe_routing_in_one_launch(ctx, orc, E, top_k, T, one):
    """A routing whose table of logits would be more than the 48 KB that one launch takes, but which brings none: one launch up to
    2^17 looks at a pair, three beyond."""
    ctx.profile_begin()
    try:
        test_mxfp4_moe_routed_follows_the_oracle(ctx, orc, 96, 64, E, top_k, T)
    finally:
        prof = ctx.profile_end()
    assert ("moe_route_lists" in prof) == one and ("moe_copy_routing" in prof) != one, sorted(prof)


@pytest.mark.parametrize("E,top_k,T", [(8, 3, 85), (8, 3, 86), (8, 4, 64), (9, 4, 65), (64, 4, 64), (65, 4, 40), (3, 3, 85), (5, 2, 120), (40, 8, 32)])
def test_mxfp4_moe_routing_beside_the_planes(ctx, orc, E, top_k, T):
    """Up to 256 pairs over up to 64 experts are routed inside the first product's planes' launch, more ahead of it: against the oracle at
    either side of both lines, and with entries that name no expert, the same bits as with them replaced."""
    import ctypes as C
    from devbuf import DevBuf
    from peregrine_amd import _ffi, mxfp4
    from test_oracle_formats_pins import _mx_expert
    hidden, inter = 96, 64
    test_mxfp4_moe_routed_follows_the_oracle(ctx, orc, hidden, inter, E, top_k, T)
    say(f"mxfp4 moe odd entries beside the planes E={E} top_k={top_k} T={T}")
    rng = np.random.default_rng(T + E)
    some = [mxfp4.Mxfp4Expert(hidden, inter, 1.702, 7.0, *_mx_expert(rng, hidden, inter), ctx=ctx) for _ in range(3)]
    tab = (C.c_void_p * E)(*[some[e % 3]._h.value for e in range(E)])
    x = rng.standard_normal((T, hidden)).astype(np.float32)
    idx = np.stack([rng.permutation(E)[:top_k] for _ in range(T)]).astype(np.int32)
    w = rng.uniform(0.2, 1.0, (T, top_k)).astype(np.float32)
    idx[rng.integers(0, T, 5), rng.integers(0, top_k, 5)] = [-1, E, 2 ** 31 - 1, -2 ** 31, idx[0, 0]]
    idx[T - 1, top_k - 1] = idx[T - 1, 0] if top_k > 1 else E
    fixed, fw = idx.copy(), w.copy()
    for t in range(T):
        taken = set()
        for k in range(top_k):
            e = int(fixed[t, k])
            if e < 0 or e >= E or e in taken:
                fixed[t, k] = e = min(set(range(E)) - taken)
                fw[t, k] = 0.0
            taken.add(e)
    assert (fixed != idx).any()

    def rows(idx, w):
        dx, di, dw, dout = DevBuf(ctx, host=x), DevBuf(ctx, host=idx), DevBuf(ctx, host=w), DevBuf(ctx, T * hidden * 4)
        _ffi.check(_ffi.lib.pg_mxfp4_moe_ffn_routed_dev(ctx.handle, dx.ptr, T, di.ptr, dw.ptr, top_k, C.cast(tab, C.POINTER(C.c_void_p)), E, dout.ptr))
        ctx.sync()
        return dout.to_host(np.float32)
    ctx.profile_begin()
    got = rows(idx, w)
    assert ("mxfp4_planes_route" in ctx.profile_end()) == (T * top_k <= 256 and E <= 64)
    np.testing.assert_array_equal(got, rows(fixed, fw))
    for ex in some:
        ex.free()


@pytest.mark.parametrize("hidden,inter,E,top_k,T", [(64, 96, 6, 6, 3), (512, 512, 200, 64, 1), (512, 96, 70, 12, 5), (64, 512, 2, 1, 9), (64, 96, 9, 4, 6), (96, 64, 5, 3, 8),
                                                   (64, 96, 8, 5, 4), (96, 64, 4, 2, 7)])
def test_mxfp4_moe_pairs_with_entries_that_name_no_expert(ctx, hidden, inter, E, top_k, T):
    """Entries out of range or named twice count as the lowest free expert with weight 0: the device entry's rows are those of the
    routing with them replaced so, in every bit, and the caller's entries stay as they were."""
    import ctypes as C
    from devbuf import DevBuf
    from peregrine_amd import _ffi, mxfp4
    from test_oracle_formats_pins import _mx_expert
    say(f"mxfp4 moe odd entries hidden={hidden} inter={inter} E={E} top_k={top_k} T={T}")
    rng = np.random.default_rng(T + E)
    some = [mxfp4.Mxfp4Expert(hidden, inter, 1.702, 7.0, *_mx_expert(rng, hidden, inter), ctx=ctx) for _ in range(min(E, 4))]
    tab = (C.c_void_p * E)(*[some[e % len(some)]._h.value for e in range(E)])
    x = rng.standard_normal((T, hidden)).astype(np.float32)
    idx = np.stack([rng.permutation(E)[:top_k] for _ in range(T)]).astype(np.int32)
    w = rng.uniform(0.2, 1.0, (T, top_k)).astype(np.float32)
    idx[0, top_k // 2] = -3
    idx[T // 2, top_k - 1] = E
    idx[T - 1, top_k - 1] = idx[T - 1, 0]
    fixed, fw = idx.copy(), w.copy()
    for t in range(T):
        taken = set()
        for k in range(top_k):
            e = int(fixed[t, k])
            if e < 0 or e >= E or e in taken:
                fixed[t, k] = e = min(set(range(E)) - taken)
                fw[t, k] = 0.0
            taken.add(e)

    def rows(idx, w):
        dx, di, dw, dout = DevBuf(ctx, host=x), DevBuf(ctx, host=idx), DevBuf(ctx, host=w), DevBuf(ctx, T * hidden * 4)
        _ffi.check(_ffi.lib.pg_mxfp4_moe_ffn_routed_dev(ctx.handle, dx.ptr, T, di.ptr, dw.ptr, top_k, C.cast(tab, C.POINTER(C.c_void_p)), E, dout.ptr))
        ctx.sync()
        assert (di.to_host(np.int32).reshape(T, top_k) == idx).all()
        return dout.to_host(np.float32).reshape(T, hidden)
    ctx.profile_begin()
    got = rows(idx, w)
    assert "mxfp4_rows_pairs" in ctx.profile_end()
    np.testing.assert_array_equal(got, rows(fixed, fw))
    for ex in some:
        ex.free()
