"""GPU parity of the matrix-core products of split weights (split.hip): every
tile (asserted by name), the ragged ends of rows, columns and K, every K-group
remainder, and infinities, NaNs and tiny values; and of the column strips
(ragged.hip).

Tolerance: rel-L2 1e-5 against the oracle, the path's bound for f32 products.
The split itself is within 2^-26 of each product; both sides round their sums.
"""
import re

import numpy as np
import pytest

import accel_amd
import oracle
from accel_amd import BF16, F16, F32, U32, workloads
from conftest import rel_l2

pytestmark = pytest.mark.gpu

F32_TOL = 1e-5
# one rounding to bf16 of an f32 result: half a unit of 8 bits is 2^-8 of a value at most
BF16_ROUND = 2.0 ** -8 + F32_TOL


def int8_run(dev, a, q, s, M, K, N, f16=False):
    ab = dev.upload(a.reshape(M, K), F16 if f16 else F32)
    qb, sb, ob = dev.upload(q.reshape(K, N)), dev.upload(s), dev.alloc((M, N), F32)
    dev.QuantMatMul(ab, qb, sb, ob)
    got = ob.numpy()
    for b in (ab, qb, sb, ob):
        b.free()
    return got


# (M, K, N): K of no whole stage, fewer stages than K groups, a ragged last
# stage; one row, one column, column pairs cut by the edge; N odd, even and
# whole blocks (which tile: TILES below)
INT8 = [(9, 1, 1), (9, 31, 33), (33, 32, 64), (10, 95, 130), (64, 257, 65), (31, 300, 2),
        (2, 1656, 1359), (130, 511, 96), (257, 1000, 1500), (100, 4100, 4004),
        (512, 1024, 8192), (2048, 260, 8190), (65, 4097, 16383)]


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("M,K,N", INT8)
def test_int8_matches_the_oracle(dev, M, K, N, f16):
    rng = np.random.default_rng(M * 31 + K * 17 + N)
    a = rng.standard_normal(M * K).astype(np.float32)
    q, s = oracle.int8_quantize((rng.standard_normal(K * N) * 0.05).astype(np.float32))
    if f16:
        a = oracle.to_f16(a)
    got = int8_run(dev, a, q, s, M, K, N, f16)
    x = (oracle.f16_to_f32(a) if f16 else a).astype(np.float64).reshape(M, K)
    w = q.astype(np.float64) * oracle.f16_to_f32(s).astype(np.float64)[np.arange(K * N) // 32]
    assert rel_l2(got, x @ w.reshape(K, N)) <= F32_TOL


# The five tiles, (32-row m-tiles, waves across the columns, K groups), and rows,
# depth and width that the cost rule gives each on the MI355X's 256 CUs, also a
# few columns either way.
TILES = [((2, 1, 8), 250, 300, 4000), ((2, 2, 4), 400, 300, 4000), ((2, 4, 2), 500, 160, 8000),
         ((1, 1, 8), 100, 300, 4000), ((1, 1, 16), 33, 300, 1000)]
TILE_IDS = ["64x64", "64x128", "64x256", "32x64", "32x32"]


def tile_of(sel):
    """The tile of a split product's launch, from its reported name."""
    found = [re.match(r"split_(?:product|grouped)_kernel<.*, (\d+), (\d+), (\d+)>", k)
             for k in sel.launches]
    return next((tuple(int(v) for v in m.groups()) for m in found if m), None)


def planned_tile(M, K, N):
    """The tile of an M x K x N product of split weights: the rule looks at the
    extents alone, so an int4 product of an even width next to N's reports it."""
    return tile_of(accel_amd.select(M, K, N + N % 2, F32))


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("more", [0, 1, 2])   # whole blocks of 32, odd, even
@pytest.mark.parametrize("tile,M,K,N", TILES, ids=TILE_IDS)
def test_int8_on_every_tile_matches_the_oracle(dev, tile, M, K, N, more, f16):
    N += more - (8 if N == 1000 else 0)       # 992 is whole blocks
    assert planned_tile(M, K, N) == tile
    test_int8_matches_the_oracle(dev, M, K, N, f16)


# Activations near the ends of the f32 range, weights of ordinary size: the
# smallest normals, subnormals (17 bits left near 2^-132) and values whose bf16
# terms' products pass the largest f32 on the way.  An f32 sum of such products
# rounds at 2^-150, far below the bound.
ENDS = [-132, -126, -120, -115, 100, 112]


def scaled_l2(got, want, e):
    return rel_l2(np.ldexp(got.astype(np.float64), -e), np.ldexp(want, -e))


@pytest.mark.parametrize("e", ENDS)
@pytest.mark.parametrize("M,K,N", [(16, 256, 128), (40, 300, 203)])
def test_int8_rows_at_the_ends_of_the_f32_range(dev, M, K, N, e):
    rng = np.random.default_rng(M + 200 + e)
    a = np.ldexp(rng.standard_normal((M, K)), e).astype(np.float32)
    q, s = oracle.int8_quantize(rng.standard_normal(K * N).astype(np.float32))
    w = q.astype(np.float64) * oracle.f16_to_f32(s).astype(np.float64)[np.arange(K * N) // 32]
    got = int8_run(dev, a, q, s, M, K, N)
    assert scaled_l2(got, a.astype(np.float64) @ w.reshape(K, N), e) <= F32_TOL


def test_int8_infinities_nans_and_the_largest_values_read_as_in_f32(dev):
    M, K, N = 40, 300, 200
    rng = np.random.default_rng(3)
    a = rng.standard_normal((M, K)).astype(np.float32)
    q, s = oracle.int8_quantize((rng.standard_normal(K * N) * 0.05).astype(np.float32))
    a[3, 7] = np.inf
    a[5, 9] = -np.inf
    a[6, 1] = np.nan
    a[8, 4] = 3.4e38            # rounds to a bf16 infinity; the product is finite
    q.reshape(K, N)[4, :] = 0
    q.reshape(K, N)[4, 50] = 1
    got = int8_run(dev, a, q, s, M, K, N)
    w = (q.astype(np.float32) * oracle.f16_to_f32(s)[np.arange(K * N) // 32]).reshape(K, N)
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ w.astype(np.float64)
    for row in (3, 5):
        k = 7 if row == 3 else 9
        inf = (w[k] != 0)
        assert np.array_equal(np.isinf(got[row]), inf)
        assert np.array_equal(np.sign(got[row][inf]), np.sign(a[row, k] * w[k][inf]))
        assert np.all(np.isnan(got[row][~inf]))
    assert np.all(np.isnan(got[6]))
    assert np.all(np.isfinite(got[8]))
    rest = np.setdiff1d(np.arange(M), (3, 5, 6))
    for row in rest:
        assert rel_l2(got[row], want[row]) <= F32_TOL, row


def test_int8_tiny_activations_keep_f32_accuracy(dev):
    # unscaled, the last bf16 term of values near 2^-115 would be a bf16 subnormal
    M, K, N = 16, 256, 128
    rng = np.random.default_rng(4)
    a = (rng.standard_normal((M, K)) * 2.0 ** -115).astype(np.float32)
    q, s = oracle.int8_quantize(rng.standard_normal(K * N).astype(np.float32))
    w = q.astype(np.float64) * oracle.f16_to_f32(s).astype(np.float64)[np.arange(K * N) // 32]
    got = int8_run(dev, a, q, s, M, K, N)
    assert rel_l2(got.astype(np.float64) * 2.0 ** 115,
                  (a.astype(np.float64) * 2.0 ** 115) @ w.reshape(K, N)) <= F32_TOL


def grouped_run(dev, form, x, w, counts, T, K, N):
    xb, wb = dev.upload(x.reshape(T, K)), dev.upload(w)
    cb, ob = dev.upload(np.array(counts, np.uint32), U32), dev.alloc((T, N), F32)
    ob.write(np.full((T, N), 7.0, np.float32))
    getattr(dev, form)(xb, wb, cb, ob)
    got = ob.numpy()
    for b in (xb, wb, cb, ob):
        b.free()
    return got


# (K, N, counts, T): one row, empty experts, blocks that end in one row, rows
# past the last segment, N odd and even, K of no whole stage
GROUPED = [(7, 1, [1], 1), (100, 33, [0, 5, 0, 65], 73), (64, 130, [1, 0, 0, 1], 3),
           (257, 64, [64, 1, 33, 0], 98), (300, 1022, [129, 3], 140), (1024, 2048, [70, 90, 60], 220),
           (32, 24000, [200, 300, 140, 1], 641), (130, 1000, [0, 0, 0], 5)]


@pytest.mark.parametrize("form", ["GroupedMatVec", "GroupedMatMul"])
@pytest.mark.parametrize("K,N,counts,T", GROUPED)
def test_grouped_f32_matches_the_oracle(dev, form, K, N, counts, T):
    E = len(counts)
    rng = np.random.default_rng(K * 31 + N)
    x = rng.standard_normal((T, K)).astype(np.float32)
    w = (rng.standard_normal((E, K, N)) * 0.05).astype(np.float32)
    got = grouped_run(dev, form, x, w, counts, T, K, N)
    at = 0
    for e, c in enumerate(counts):
        if c:
            want = x[at:at + c].astype(np.float64) @ w[e].astype(np.float64)
            assert rel_l2(got[at:at + c], want) <= F32_TOL, e
        at += c
    assert np.all(got[at:] == (0 if form == "GroupedMatVec" else 7.0))


# The same for the grouped products: half of the tokens in one expert, the depth
# whole groups whatever the width.
GROUPED_TILES = [((2, 1, 8), 2, 128, 256, 4000), ((2, 2, 4), 8, 256, 256, 4000),
                 ((2, 4, 2), 4, 640, 128, 4000), ((1, 1, 8), 2, 90, 256, 4000),
                 ((1, 1, 16), 2, 6, 512, 1000)]


@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("tile,E,T,K,N", GROUPED_TILES, ids=TILE_IDS)
def test_grouped_products_on_every_tile_match_the_oracle(dev, tile, E, T, K, N, odd):
    rng = np.random.Generator(np.random.PCG64(T + odd))
    counts = [T // 2] + [(T - T // 2) // (E - 1)] * (E - 1)
    counts[-1] += T - sum(counts)
    # int4 experts of an even width, whose report names the tile
    p, s, z, w = int4_weights(rng, E * K, N + 2 * odd)
    x = rng.standard_normal((T, K)).astype(np.float32)
    xb, wd = dev.upload(x), dev.upload_int4(p, s, z, w.size)
    cb, ob = dev.upload(np.array(counts, np.uint32), U32), dev.alloc((T, N + 2 * odd), F32)
    dev.Int4GroupedMatMul(xb, wd, E, cb, ob)
    got4, sel = ob.numpy(), dev.last_selection()
    for b in (xb, wd, cb, ob):
        b.free()
    assert tile_of(sel) == tile, sel
    # f32 experts: the same rule, the same extents (odd: one column less)
    wf = (rng.standard_normal((E, K, N + odd)) * 0.05).astype(np.float32)
    got = grouped_run(dev, "GroupedMatMul", x, wf, counts, T, K, N + odd)
    w, at = w.reshape(E, K, N + 2 * odd), 0
    for e, c in enumerate(counts):
        xe = x[at:at + c].astype(np.float64)
        assert rel_l2(got4[at:at + c], xe @ w[e]) <= F32_TOL, e
        assert rel_l2(got[at:at + c], xe @ wf[e].astype(np.float64)) <= F32_TOL, e
        at += c


# (exponent of the rows, of the weights)
@pytest.mark.parametrize("ex,ew", [(e, 0) for e in ENDS] + [(0, e) for e in ENDS] + [(-124, 100), (60, 52)])
def test_grouped_f32_at_the_ends_of_the_f32_range(dev, ex, ew):
    E, T, K, N = 2, 40, 256, 96
    rng = np.random.default_rng(13)
    x = np.ldexp(rng.standard_normal((T, K)), ex).astype(np.float32)
    w = np.ldexp(rng.standard_normal((E, K, N)), ew).astype(np.float32)
    got = grouped_run(dev, "GroupedMatMul", x, w, [20, 20], T, K, N)
    for e in range(E):
        rows = slice(20 * e, 20 * e + 20)
        want = x[rows].astype(np.float64) @ w[e].astype(np.float64)
        assert scaled_l2(got[rows], want, ex + ew) <= F32_TOL, e


@pytest.mark.parametrize("form", ["GroupedMatVec", "GroupedMatMul"])
@pytest.mark.parametrize("counts", [[3, 0xFFFFFFFF, 4, 2], [6, 0xFFFFFFFA, 6], [9, 4]])
def test_grouped_f32_offsets_that_wrap_or_run_past_the_rows(dev, form, counts):
    E, T, K, N = len(counts), 8, 96, 70
    rng = np.random.default_rng(11)
    x = rng.standard_normal((T, K)).astype(np.float32)
    w = rng.standard_normal((E, K, N)).astype(np.float32)
    got = grouped_run(dev, form, x, w, counts, T, K, N)
    off = np.concatenate([[0], np.cumsum(np.array(counts, np.uint64)) & 0xFFFFFFFF])
    for t in range(T):
        e = int(np.sum(off[1:] <= t))
        covered = e < E and off[e] <= t < min(off[e + 1], T)
        if e < E and (covered or form == "GroupedMatVec"):
            want = x[t].astype(np.float64) @ w[e].astype(np.float64)
            assert rel_l2(got[t], want) <= F32_TOL, t
        else:
            assert np.all(got[t] == (0 if form == "GroupedMatVec" else 7.0)), t


def test_grouped_f32_infinite_and_nan_weights_read_as_in_f32(dev):
    E, T, K, N = 2, 40, 64, 96
    rng = np.random.default_rng(12)
    x = np.abs(rng.standard_normal((T, K))).astype(np.float32) + 0.5
    w = rng.standard_normal((E, K, N)).astype(np.float32)
    w[0, 3, 5], w[1, 4, 6], w[1, 5, 7] = np.inf, -np.inf, np.nan
    got = grouped_run(dev, "GroupedMatMul", x, w, [20, 20], T, K, N)
    assert np.all(got[:20, 5] == np.inf) and np.all(got[20:, 6] == -np.inf)
    assert np.all(np.isnan(got[20:, 7]))
    got[:20, 5] = got[20:, 6] = got[20:, 7] = 0
    assert np.all(np.isfinite(got))


def int4_run(dev, a, p, s, z, M, K, N, bf16=False, form="Int4MatMul", bias=None):
    ab = dev.upload(a, BF16 if bf16 else F32)
    wd = dev.upload_int4(p, s, z, K * N)
    ob = dev.alloc((M, N) if a.ndim == 2 else (N,), BF16 if bf16 else F32)
    bb = dev.upload(bias) if bias is not None else None
    if form == "Int4Linear":
        dev.Int4Linear(ab, wd, bb, ob)
    else:
        getattr(dev, form)(ab, wd, ob)
    got, launches = ob.numpy(), dev.last_selection().launches
    for b in (ab, ob, wd, bb):
        if b:
            b.free()
    return (workloads.bf16_to_f32(got) if bf16 else got), launches


def int4_weights(rng, K, N):
    p, s, z = workloads.fast_int4(K, N, rng)
    s, z = s.copy(), z.copy()
    s[1], z[1] = 0, oracle.to_f16(np.array([0.75], np.float32))[0]     # a constant group
    z[-1] = oracle.to_f16(np.array([-900.0], np.float32))[0]           # far from zero
    w = oracle.int4_dequantize(p, s, z, K * N).astype(np.float64).reshape(K, N)
    return p, s, z, w


# (K, N): every N mod 8 (the words' alignments), strips that end in one column
# and in whole, K below, at and past the row phases and their batches
RAGGED = [(32, 65), (33, 70), (128, 66), (130, 65), (511, 570), (512, 571), (513, 572), (200, 61 + 64), (1000, 1001),
          (4096, 1004), (129, 4095), (777, 30 * 56), (300, 30 * 56 + 1), (2048, 126),
          # the strips of 120 and of 248 columns
          (1000, 14393), (385, 30600), (130, 30723), (700, 31000)]


@pytest.mark.parametrize("K,N", RAGGED)
def test_int4_matvec_of_any_width_matches_the_oracle(dev, K, N):
    rng = np.random.Generator(np.random.PCG64(K * 31 + N))
    p, s, z, w = int4_weights(rng, K, N)
    for M, bf16 in ((1, False), (1, True), (2, False), (3, True), (4, False)):
        x = rng.standard_normal((M, K)).astype(np.float32)
        bits = workloads.bf16_bits(x)
        want = (workloads.bf16_to_f32(bits) if bf16 else x).astype(np.float64) @ w
        if M == 1 and not bf16:
            got, launches = int4_run(dev, x[0], p, s, z, 1, K, N, form="Int4MatVec")
            again, _ = int4_run(dev, x[0], p, s, z, 1, K, N, form="Int4MatVecNoAlloc")
            assert np.array_equal(got, again)
        else:
            got, launches = int4_run(dev, bits if bf16 else x, p, s, z, M, K, N, bf16)
        assert launches[0].startswith("ragged_rows_kernel<"), launches
        assert rel_l2(got, want if M > 1 or bf16 else want[0]) <= (4e-3 if bf16 else F32_TOL), (M, bf16)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M,K,N", [(1, 33, 65), (2, 130, 203), (4, 511, 1001), (3, 130, 14401)])
def test_int4_linear_of_few_rows_of_any_width_adds_the_bias(dev, M, K, N, bf16):
    rng = np.random.Generator(np.random.PCG64(M * 31 + N))
    p, s, z, w = int4_weights(rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float32)
    bias = (100 * rng.standard_normal(N)).astype(np.float32)
    bits = workloads.bf16_bits(x)
    run = lambda b: int4_run(dev, bits if bf16 else x, p, s, z, M, K, N, bf16, "Int4Linear", b)  # noqa: E731
    got, launches = run(bias)
    assert launches[0].startswith("ragged_rows_kernel<"), launches
    if not bf16:
        # one f32 addition to what the product alone stores
        assert np.array_equal(got, run(None)[0] + bias)
    want = (workloads.bf16_to_f32(bits) if bf16 else x).astype(np.float64) @ w + bias
    assert rel_l2(got, want) <= (BF16_ROUND if bf16 else F32_TOL)


def test_int4_matvec_of_any_width_infinities_and_nans(dev):
    K, N = 300, 203
    rng = np.random.Generator(np.random.PCG64(9))
    p, s, z, w = int4_weights(rng, K, N)
    x = rng.standard_normal(K).astype(np.float32)
    x[299] = np.inf           # the last row: its words end the planes
    got, _ = int4_run(dev, x, p, s, z, 1, K, N, form="Int4MatVec")
    assert np.array_equal(np.isinf(got), w[299] != 0)
    x[299], x[0] = 1, np.nan
    got, _ = int4_run(dev, x, p, s, z, 1, K, N, form="Int4MatVec")
    assert np.all(np.isnan(got))


@pytest.mark.parametrize("M", [1, 3])
def test_int4_rows_whose_scaled_activation_overflows_stay_finite(dev, M):
    # 1e36 x 4096 overflows, but where the code is the zero point the weight is 0
    K, N = 300, 203
    rng = np.random.Generator(np.random.PCG64(10))
    p, s, z, _ = int4_weights(rng, K, N)
    s[8], z[8] = oracle.to_f16(np.array([4096.0, 8.0], np.float32))   # of row 5: columns 9..136
    w = oracle.int4_dequantize(p, s, z, K * N).astype(np.float64).reshape(K, N)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[M - 1, 5] = 1e36
    got, launches = int4_run(dev, x, p, s, z, M, K, N)
    assert launches[0].startswith("ragged_rows_kernel<"), launches
    want = x.astype(np.float64) @ w
    over = np.abs(want) > 3.5e38
    assert over.any() and np.sum(w[5, 9:137] == 0) > 0
    assert np.array_equal(np.isinf(got), over)
    bound = K * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w))   # of K f32 roundings
    assert np.all(np.abs(got - want)[~over] <= bound[~over])


@pytest.mark.parametrize("M,bf16", [(1, False), (2, True), (4, False)])
@pytest.mark.parametrize("e,scale,zero", [(-124, 2.0 ** -14, -500.0), (-115, 2.0 ** -14, -500.0),
                                          (-126, 0.25, 7.3), (100, 0.25, 7.3), (112, 0.25, 7.3)])
def test_int4_rows_of_any_width_at_the_ends_of_the_f32_range(dev, M, bf16, e, scale, zero):
    # an activation times its scale leaves f32's normal numbers before its
    # products with the weights, scale (code - zero), do
    K, N = 1000, 203
    rng = np.random.Generator(np.random.PCG64(15))
    p, _, _, _ = int4_weights(rng, K, N)
    groups = -(-K * N // 128)
    s, z = (oracle.to_f16(np.full(groups, v, np.float32)) for v in (scale, zero))
    w = oracle.int4_dequantize(p, s, z, K * N).astype(np.float64).reshape(K, N)
    x = np.ldexp(rng.standard_normal((M, K)), e).astype(np.float32)
    bits = workloads.bf16_bits(x)
    got, launches = int4_run(dev, bits if bf16 else x, p, s, z, M, K, N, bf16)
    assert launches[0].startswith("ragged_rows_kernel<"), launches
    want = (workloads.bf16_to_f32(bits) if bf16 else x).astype(np.float64) @ w
    assert scaled_l2(got, want, e) <= (BF16_ROUND if bf16 else F32_TOL)


# (M, K, N): N odd, even and whole groups (there K % 64 != 0 keeps the int4
# tiles off), K of no whole stage, and one row past the few-rows kernel
INT4 = [(5, 128, 65), (6, 129, 64), (9, 32, 66), (40, 47, 333), (33, 200, 1001), (17, 511, 130), (64, 1000, 999),
        (100, 4100, 4004), (40, 136, 384), (70, 2090, 256), (513, 260, 8190), (300, 1026, 4098),
        (65, 130, 16391)]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("M,K,N", INT4)
def test_int4_rows_of_any_extents_match_the_oracle(dev, M, K, N, bf16):
    rng = np.random.Generator(np.random.PCG64(M * 31 + K * 17 + N))
    p, s, z, w = int4_weights(rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    bits = workloads.bf16_bits(x)
    got, launches = int4_run(dev, bits if bf16 else x, p, s, z, M, K, N, bf16, "Int4Linear", bias)
    assert launches[0].startswith("split_product_kernel<"), launches
    want = (workloads.bf16_to_f32(bits) if bf16 else x).astype(np.float64) @ w + bias
    # bf16: one rounding of the result (2^-8 at most, 2^-9.2 in the norm of many values)
    assert rel_l2(got, want) <= (2.0 ** -9 if bf16 else F32_TOL)


# Even widths and whole groups (where the 64-column tiles start halfway through
# one) on every tile; odd widths take the 32-row tiles alone.
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("form", ["odd", "even", "groups"])
@pytest.mark.parametrize("tile,M,K,N", TILES, ids=TILE_IDS)
def test_int4_on_every_tile_matches_the_oracle(dev, tile, M, K, N, form, bf16):
    N = {"odd": N + 1, "even": N + 2, "groups": (N + 64) // 128 * 128}[form]
    sel = accel_amd.select(M, K, N, BF16 if bf16 else F32)
    want = tile if form != "odd" or tile == (1, 1, 16) else (1, 1, 8)
    assert tile_of(sel) == want, sel
    test_int4_rows_of_any_extents_match_the_oracle(dev, M, K, N, bf16)


@pytest.mark.parametrize("e", ENDS)
def test_int4_rows_of_any_extents_at_the_ends_of_the_f32_range(dev, e):
    M, K, N = 20, 300, 203
    rng = np.random.Generator(np.random.PCG64(14))
    p, _, _, _ = int4_weights(rng, K, N)
    groups = -(-K * N // 128)
    s = oracle.to_f16(np.full(groups, 0.25, np.float32))
    z = oracle.to_f16(rng.uniform(0, 15, groups).astype(np.float32))
    w = oracle.int4_dequantize(p, s, z, K * N).astype(np.float64).reshape(K, N)
    x = np.ldexp(rng.standard_normal((M, K)), e).astype(np.float32)
    got, launches = int4_run(dev, x, p, s, z, M, K, N)
    assert launches[0].startswith("split_product_kernel<"), launches
    assert scaled_l2(got, x.astype(np.float64) @ w, e) <= F32_TOL


def test_int4_rows_of_any_extents_infinities(dev):
    M, K, N = 20, 300, 203
    rng = np.random.Generator(np.random.PCG64(10))
    p, s, z, w = int4_weights(rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[2, 299], x[3, 0] = -np.inf, np.nan
    got, _ = int4_run(dev, x, p, s, z, M, K, N)
    assert np.array_equal(got[2] == -np.inf, w[299] > 0)
    assert np.array_equal(got[2] == np.inf, w[299] < 0)
    assert np.all(np.isnan(got[3])) and np.all(np.isfinite(np.delete(got, (2, 3), 0)))


@pytest.mark.parametrize("form", ["Int4GroupedMatVec", "Int4GroupedMatMul"])
@pytest.mark.parametrize("K,N,counts,T", [(128, 33, [3, 0, 40], 45), (256, 130, [1, 70], 71),
                                          (160, 4, [2, 3], 6), (384, 1002, [100, 0xFFFFFFFF, 30], 120)])
def test_int4_grouped_of_any_width_matches_the_oracle(dev, form, K, N, counts, T):
    E = len(counts)
    rng = np.random.Generator(np.random.PCG64(K + N))
    p, s, z, w = int4_weights(rng, E * K, N)
    w = w.reshape(E, K, N)
    x = rng.standard_normal((T, K)).astype(np.float32)
    xb, wd = dev.upload(x), dev.upload_int4(p, s, z, E * K * N)
    cb, ob = dev.upload(np.array(counts, np.uint32), U32), dev.alloc((T, N), F32)
    ob.write(np.full((T, N), 7.0, np.float32))
    getattr(dev, form)(xb, wd, E, cb, ob)
    got, launches = ob.numpy(), dev.last_selection().launches
    for b in (xb, wd, cb, ob):
        b.free()
    assert any(k.startswith("split_grouped_kernel<Int4W") for k in launches), launches
    off = np.concatenate([[0], np.cumsum(np.array(counts, np.uint64)) & 0xFFFFFFFF])
    for t in range(T):
        e = int(np.sum(off[1:] <= t))
        if e < E and (form == "Int4GroupedMatVec" or off[e] <= t < min(off[e + 1], T)):
            assert rel_l2(got[t], x[t].astype(np.float64) @ w[e]) <= F32_TOL, t
        else:
            assert np.all(got[t] == (0 if form == "Int4GroupedMatVec" else 7.0)), t


# Past the tiles' widths (N <= 2^24) the kernels of one lane, or one small f32
# tile, per element still run.

def test_int4_grouped_past_the_tiles_widths_says_so_and_matches_the_oracle(dev):
    E, T, K, N = 2, 3, 2, (1 << 24) + 64
    rng = np.random.Generator(np.random.PCG64(16))
    groups = E * K * N // 128
    p = rng.integers(0, 1 << 32, E * K * N // 8, dtype=np.uint64).astype(np.uint32)
    s = oracle.to_f16(rng.uniform(0.01, 0.02, groups).astype(np.float32))
    z = oracle.to_f16(rng.uniform(0, 15, groups).astype(np.float32))
    w = oracle.int4_dequantize(p, s, z, E * K * N).reshape(E, K, N)
    x = rng.standard_normal((T, K)).astype(np.float32)
    xb, wd = dev.upload(x), dev.upload_int4(p, s, z, E * K * N)
    cb, ob = dev.upload(np.array([2, 1], np.uint32), U32), dev.alloc((T, N), F32)
    dev.Int4GroupedMatMul(xb, wd, E, cb, ob)
    got, sel = ob.numpy(), dev.last_selection()
    for b in (xb, wd, cb, ob):
        b.free()
    assert sel.launches[-1].startswith("grouped_f32_kernel<true>"), sel
    assert "one lane per" in sel.reason and "split" not in sel.reason, sel
    assert any("tiles of split weights" in r for r in sel.rejected), sel
    for t, e in enumerate((0, 0, 1)):
        assert rel_l2(got[t], x[t].astype(np.float64) @ w[e]) <= F32_TOL, t


@pytest.mark.parametrize("f16", [False, True])
def test_int8_past_the_tiles_widths_matches_the_oracle(dev, f16):
    test_int8_matches_the_oracle(dev, 2, 3, (1 << 24) + 1, f16)


def test_grouped_f32_past_the_tiles_widths_matches_the_oracle(dev):
    for form in ("GroupedMatVec", "GroupedMatMul"):
        test_grouped_f32_matches_the_oracle(dev, form, 2, (1 << 24) + 1, [2, 1], 4)


@pytest.mark.parametrize("n", [2047, 2048, 2049, 16384 + 1920, 3 * 2048 + 128 * 5 + 77])
def test_packer_waves_of_sixteen_groups_are_bit_exact(dev, n):
    """Whole waves beside single groups, and waves that leave the fast path:
    a NaN or infinity anywhere, a -0.0 minimum, constant groups, ranges whose
    f16 scale is zero, subnormal or infinite."""
    rng = np.random.default_rng(n)
    base = (rng.standard_normal(n) * 0.02).astype(np.float32)
    odd = base.copy()
    odd[-128:] = 0.0
    odd[: 128] = np.abs(odd[: 128])
    odd[5] = -0.0
    odd[300] = np.nan
    odd[1023] = np.inf
    scales = np.repeat(10.0 ** rng.integers(-12, 30, n // 128 + 1), 128)[:n]
    for w in (base, odd, np.maximum(base, 0), (base * scales).astype(np.float32),
              np.full(n, -3.25, np.float32), np.zeros(n, np.float32)):
        wb = dev.upload(w)
        pb, sb = dev.alloc(((n + 7) // 8,), U32), dev.alloc(((n + 127) // 128,), F16)
        zb = dev.alloc(((n + 127) // 128,), F16)
        dev.int4_quantize(wb, n, pb, sb, zb)
        for got, want in zip((pb, sb, zb), oracle.int4_quantize(w)):
            assert np.array_equal(got.numpy(), want)
        for b in (wb, pb, sb, zb):
            b.free()
