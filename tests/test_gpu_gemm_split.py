"""GPU checks of the split GEMM tiles (gemm_split.hip): f32 products from six
bf16 MFMA products of exact three-way splits, against 64-bit sums.

Bound per element: with S = sum_p |a_p b_p|, the three products left out are
below 3 * 2^-24 S; the matrix core rounds the running sum once per product
group of 16 k, six groups per 16 k, each below 2^-23 S (it may truncate); a K
split adds at most 16 partials, a rounding of 2^-24 each. So |err| <=
(6 * ceil(k / 16) + 16) * 2^-23 * S.
"""
import ctypes

import numpy as np
import pytest

import midman_hip as mh

pytestmark = pytest.mark.gpu

# (m, k, n) with row, column and K remainders, and the tile and K splits that
# the choice in gemm.hip gives each on 256 CUs (test_plans holds it to that)
PLANS = [
    ("256x128, K tail", 3900, 100, 4000, 1),
    ("256x128, whole steps", 2050, 64, 4100, 1),
    ("256x256 in 3 splits", 1000, 2050, 4100, 3),
    ("128x128, 2 wave groups, odd step and tail", 1000, 777, 3071, 1),
    ("64x64, 4 wave groups, 2 odd steps and a tail", 1003, 1517, 770, 1),
    ("128x64, an odd step", 2000, 528, 1001, 1),
    ("64x64, 4 wave groups, 3 odd steps and a tail", 1030, 569, 515, 1),
    ("64x64 in 10 splits", 300, 5003, 301, 10),
    ("128x128 in 3 splits", 767, 1598, 1373, 3),
    ("64x64 in 16 splits", 130, 9001, 257, 16),
    ("256x128, few steps and a tail", 2300, 50, 2301, 1),
    ("256x256, K tail", 3344, 66, 3105, 1),
    ("256x128 in 11 splits", 134, 3670, 2208, 11),
    ("128x64 in 6 splits", 341, 899, 876, 6),
    ("128x64, fewer whole steps than wave groups", 32768, 31, 60, 1),
]
SHAPES = [p[:4] for p in PLANS]
# small products, 32x32 tiles with K split over waves and workgroups: the K
# around a split's 8 and 16 steps, more than one step per wave, more tiles than
# CUs, rows that are not 16-byte aligned (summed by fp32 MFMAs: one rounding
# of at most 2^-24 of the absolute sum per value, and one per split)
SMALL = [(33, 255, 31), (64, 512, 96), (64, 513, 96), (96, 1024, 96), (128, 2016, 384),
         (32, 8192, 32), (2368, 3480, 32), (512, 1600, 320), (1435, 295, 187), (560, 1168, 174),
         (92, 1175, 135)]


def plan(ctx, form, m, k, n, accumulate=0):
    """(rows, columns, K splits) of the tiles a product of 16-byte aligned operands takes."""
    out, x = (ctypes.c_int32 * 3)(), ctx.empty((4,))
    at = ctypes.c_void_p(x.ptr)
    mh.check(mh.lib().mmh_test_gemm_plan(
        ctypes.c_int64(ctx.handle), {"nn": 0, "nt": 1, "tn": 2}[form], at, at, at, ctypes.c_int64(m),
        ctypes.c_int64(k), ctypes.c_int64(n), accumulate, out))
    x.free()
    return tuple(out)


@pytest.mark.parametrize("form", ["nn", "nt", "tn"])
def test_plans(ctx, form):
    if ctx.device_info()[1] != 256:
        pytest.skip("the plans are those of 256 CUs")
    for what, m, k, n, splits in PLANS:
        rows, cols = (int(x) for x in what.replace(",", " ").split()[0].split("x"))
        assert plan(ctx, form, m, k, n) == (rows, cols, splits), what
        assert plan(ctx, form, m, k, n, 1)[:2] == ((rows, cols) if k > 32 else (64, 64)), what
    assert all(plan(ctx, form, m, k, n)[:2] == (32, 32) for m, k, n in SMALL)


def run(ctx, form, a, b, c0=None):
    m, k, n = a.shape[0], a.shape[1], b.shape[1]
    A = ctx.to_device(np.ascontiguousarray(a.T) if form == "tn" else a)
    B = ctx.to_device(np.ascontiguousarray(b.T) if form == "nt" else b)
    C = ctx.to_device(c0) if c0 is not None else ctx.empty((m, n))
    mh.gemm(ctx, form, A, B, C, m, k, n, accumulate=c0 is not None)
    out = C.numpy()
    for x in (A, B, C):
        x.free()
    return out


def check(out, a, b, c0=None):
    want = a.astype(np.float64) @ b.astype(np.float64)
    size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    k = a.shape[1]
    bound = (6 * -(-k // 16) + 16) * 2.0**-23 * size + 2.0**-140
    if c0 is not None:
        want = want + c0
        bound = bound + 2.0**-23 * (np.abs(c0) + size)
    worst = float(np.max(np.abs(out - want) / bound))
    print(f"  max err / bound {worst:.3g}", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("what,m,k,n", SHAPES, ids=[s[0] for s in SHAPES])
@pytest.mark.parametrize("form", ["nn", "nt", "tn"])
def test_tile_edges(ctx, what, m, k, n, form):
    print(f"\n[gemm split] {what}: {form} {m}x{k}x{n}", flush=True)
    r = np.random.default_rng(m + k + n)
    a = r.standard_normal((m, k), dtype=np.float32)
    b = r.standard_normal((k, n), dtype=np.float32)
    c0 = r.standard_normal((m, n), dtype=np.float32)
    check(run(ctx, form, a, b), a, b)
    check(run(ctx, form, a, b, c0), a, b, c0)


@pytest.mark.parametrize("what,m,k,n", SHAPES, ids=[s[0] for s in SHAPES])
@pytest.mark.parametrize("lo,hi", [(-60, 60), (-126, -90), (100, 126)])
def test_every_exponent(ctx, what, m, k, n, lo, hi):
    # magnitudes from 2^lo to 2^hi on one side and their reciprocals' range on
    # the other: pieces that would be subnormal in bf16 (below 2^-102) and
    # values above its largest finite one take the fp32 products
    print(f"\n[gemm split] {what}: exponents {lo}..{hi}, {m}x{k}x{n}", flush=True)
    r = np.random.default_rng(m * 3 + k + hi)
    signs = lambda s: r.choice(np.float32([-1, 1]), s)  # noqa: E731
    mant = lambda s: r.uniform(1, 2, s).astype(np.float32)  # noqa: E731
    a = signs((m, k)) * np.ldexp(mant((m, k)), r.integers(lo, hi + 1, (m, k))).astype(np.float32)
    span = (-hi, -lo) if lo > -100 and hi < 100 else ((0, 20) if hi < 0 else (-40, -20))
    b = signs((k, n)) * np.ldexp(mant((k, n)), r.integers(span[0], span[1] + 1, (k, n))).astype(np.float32)
    check(run(ctx, "nn", a, b), a, b)


@pytest.mark.parametrize("what,m,k,n", SHAPES, ids=[s[0] for s in SHAPES])
@pytest.mark.parametrize("form", ["nn", "nt", "tn"])
def test_special_values(ctx, what, m, k, n, form):
    # inf, NaN, the largest float, subnormals and -0 in single rows, columns
    # and the last k of integer operands: exact sums, so the bits are the
    # scalar rules' (float64 arithmetic rounded once)
    print(f"\n[gemm split] special values, {what}: {form} {m}x{k}x{n}", flush=True)
    r = np.random.default_rng(k)
    a = r.integers(-3, 4, (m, k)).astype(np.float32)
    b = r.integers(-3, 4, (k, n)).astype(np.float32)
    a[1, k - 1], a[m - 1, 0] = np.inf, np.nan
    b[k - 1, n - 1] = -np.inf
    big = np.finfo(np.float32).max
    a[m // 2], b[:, n // 2] = 0.0, 0.0
    a[m // 2, 0], b[0, n // 2] = big, 1.0
    tiny = np.float32(2.0**-149)
    a[m // 3] = 0.0
    a[m // 3, k // 2] = 3 * tiny
    a[m // 4] = -0.0
    c0 = np.zeros((m, n), np.float32)
    c0[m // 4] = -0.0
    with np.errstate(invalid="ignore", over="ignore"):
        want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    out = run(ctx, form, a, b)
    assert np.array_equal(out, want, equal_nan=True)
    fin = np.isfinite(want)
    acc = run(ctx, form, a, b, c0)
    assert np.array_equal(acc[fin], (want + c0)[fin])
    # a row of -0 times positives keeps C's -0
    b2 = np.abs(np.where(np.isfinite(b), b, 1)).astype(np.float32) + 1
    acc = run(ctx, form, a, b2, c0)
    assert np.all(np.signbit(acc[m // 4])) and np.all(acc[m // 4] == 0.0)


@pytest.mark.parametrize("what,m,k,n", SHAPES, ids=[s[0] for s in SHAPES])
def test_tiny_values_cost_nothing(ctx, what, m, k, n):
    # a row of values down to the smallest subnormal, and columns scaled below
    # 2^-102: the other rows keep their bits, so no tile is formed a second way
    print(f"\n[gemm split] tiny values, {what}: {m}x{k}x{n}", flush=True)
    r = np.random.default_rng(m + n)
    a = r.standard_normal((m, k), dtype=np.float32)
    b = r.standard_normal((k, n), dtype=np.float32)
    plain = run(ctx, "nn", a, b)
    t = a.copy()
    t[::32] *= np.float32(2.0) ** r.integers(-149, -100, (len(t[::32]), k)).astype(np.float32)
    out = run(ctx, "nn", t, b)
    rest = np.arange(m) % 32 != 0
    assert np.array_equal(out[rest].view(np.uint32), plain[rest].view(np.uint32))
    check(out, t, b)
    c = np.ldexp(b, np.where(np.arange(n) % 2, -125, 0)).astype(np.float32)
    out = run(ctx, "nn", a, c)
    assert np.array_equal(out[:, ::2].view(np.uint32), plain[:, ::2].view(np.uint32))
    check(out, a, c)


# (a K of one step of 32 accumulates on the fp32 64x64 tiles)
@pytest.mark.parametrize("what,m,k,n", [s for s in SHAPES if s[2] > 32], ids=[s[0] for s in SHAPES if s[2] > 32])
@pytest.mark.parametrize("form", ["nn", "nt", "tn"])
def test_accumulated_zeros_cost_nothing(ctx, what, m, k, n, form):
    # rows that are zero over a split's k (padded tokens): its partial sums there
    # are zero, and what is added to a C of +0 has the bits of the plain product,
    # so no tile is formed a second way for the sign of a zero that nothing shows
    print(f"\n[gemm split] accumulated zeros, {what}: {form} {m}x{k}x{n}", flush=True)
    r = np.random.default_rng(m * n)
    a = r.standard_normal((m, k), dtype=np.float32)
    b = r.standard_normal((k, n), dtype=np.float32)
    a[::2, : k // 4 + 1] = 0
    a[::2, -(k // 4) :] = 0
    out = run(ctx, form, a, b, np.zeros((m, n), np.float32))
    assert np.array_equal(out, run(ctx, form, a, b))
    # beside a -0 of C a split's zeros keep their sign, and rows of -0 leave it
    c0 = np.where(np.arange(m)[:, None] % 4 == 0, np.float32(-0.0), np.float32(1.0)) * np.ones((1, n), np.float32)
    a[::4] = -0.0
    out = run(ctx, form, a, np.abs(b) + 1, c0)
    assert np.all(np.signbit(out[::4])) and np.all(out[::4] == 0)


def f32_sums(a, b, block):
    """The product by f32 sums in order over blocks of k, the blocks' sums in order."""
    total = None
    for k0 in range(0, a.shape[1], block):
        s = np.zeros((a.shape[0], b.shape[1]), np.float32)
        for k in range(k0, min(k0 + block, a.shape[1])):
            s += a[:, k, None] * b[k]
        total = s if total is None else total + s
    return total


# K of a few steps, whose f32 sums round seldom (in order over K here), and shapes
# of fewer 128x128 tiles than CUs, which had blocks of 32 on the 32x32 tiles
@pytest.mark.parametrize("m,n,k,block", [(2050, 4100, k, k) for k in (1, 2, 5, 16, 17, 31, 32, 40)]
                         + [(1472, 1091, 256, 32), (354, 4800, 256, 32), (300, 3456, 320, 32)])
def test_no_further_off_than_f32_sums(ctx, m, n, k, block):
    print(f"\n[gemm split] error of {m}x{k}x{n}", flush=True)
    r = np.random.default_rng(k)
    a, b = r.standard_normal((m, k), dtype=np.float32), r.standard_normal((k, n), dtype=np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    rel = lambda x: np.linalg.norm(x - want) / np.linalg.norm(want)  # noqa: E731
    got, ref = rel(run(ctx, "nn", a, b)), rel(f32_sums(a, b, block))
    print(f"  {got:.3g}, f32 sums {ref:.3g}", flush=True)
    assert got <= 1.02 * ref


@pytest.mark.parametrize("m,k,n", [(53, 719, 3584), (128, 602, 1984), (1239, 768, 192)])
def test_small_product_precision(ctx, m, k, n):
    # f32 sums over the 32 k of a step, the steps' sums in pairs
    print(f"\n[gemm K split] error of {m}x{k}x{n}", flush=True)
    r = np.random.default_rng(k)
    a, b = r.standard_normal((m, k), dtype=np.float32), r.standard_normal((k, n), dtype=np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    steps = [f32_sums(a[:, i:i + 32], b[i:i + 32], 32) for i in range(0, k, 32)]
    while len(steps) > 1:
        steps = [x + y for x, y in zip(steps[::2], steps[1::2])] + steps[len(steps) & ~1:]
    rel = lambda x: np.linalg.norm(x - want) / np.linalg.norm(want)  # noqa: E731
    got, ref = rel(run(ctx, "nn", a, b)), rel(steps[0])
    print(f"  {got:.3g}, f32 sums in pairs {ref:.3g}", flush=True)
    assert got <= 1.05 * ref


@pytest.mark.parametrize("m,k,n", SMALL)
@pytest.mark.parametrize("form", ["nn", "nt", "tn"])
def test_small_product_splits(ctx, m, k, n, form):
    print(f"\n[gemm K split] {form} {m}x{k}x{n}", flush=True)
    r = np.random.default_rng(m + k + n)
    a, b = r.standard_normal((m, k), dtype=np.float32), r.standard_normal((k, n), dtype=np.float32)
    c0 = r.standard_normal((m, n), dtype=np.float32)
    for c in (None, c0):
        out = run(ctx, form, a, b, c)
        want = a.astype(np.float64) @ b.astype(np.float64) + (0 if c is None else c)
        size = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64) + (0 if c is None else np.abs(c))
        worst = float((np.abs(out - want) / ((k + 64) * 2.0**-24 * size)).max())
        print(f"  max err / bound {worst:.3g}", flush=True)
        assert worst <= 1.0
