"""GPU checks of the split-bf16 attention forward (attention_split.hip: heads
of 64 and 128) against 64-bit softmax attention.

Bound: a score is a sum of hd products whose six parts are each rounded into
the sum (6 * hd / 16 roundings below 2^-23 of the absolute sum, here at most
~6 sqrt(hd) times the scale: 2e-5), so a probability is off by at most ~2e-5 of
itself; the output is a weighted mean of V with weights of that accuracy:
|err| <= 4e-5 max|v|, measured two orders below.
"""
import numpy as np
import pytest

import midman_hip as mh

pytestmark = pytest.mark.gpu


def reference(q, k, v):
    B, H, T, hd = q.shape
    out = np.empty(q.shape)
    mask = np.tril(np.ones((T, T), bool))
    for b in range(B):
        for h in range(H):
            j = h // (H // k.shape[1])
            s = q[b, h].astype(np.float64) @ k[b, j].astype(np.float64).T / np.sqrt(hd)
            s = np.where(mask, s, -np.inf)
            e = np.exp(s - s.max(-1, keepdims=True))
            with np.errstate(invalid="ignore"):
                out[b, h] = (e / e.sum(-1, keepdims=True)) @ v[b, j].astype(np.float64)
    return out


def attend(ctx, q, k, v):
    dev = [ctx.to_device(x) for x in (q, k, v)]
    return mh.causal_attention(ctx, *dev).numpy()


def inputs(B, H, Hkv, T, hd, seed):
    r = np.random.default_rng(seed)
    f = lambda h: r.standard_normal((B, h, T, hd), dtype=np.float32)  # noqa: E731
    return f(H), f(Hkv), f(Hkv)


# heads of 64 take this kernel from one 128-row block per CU on (256 blocks); short
# last blocks (up to 112 or 64 rows of one block, 56 of two or three) the 16-row one
@pytest.mark.parametrize("B,H,Hkv,hd", [(1, 4, 2, 128), (16, 16, 8, 64)])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 64, 65, 96, 97, 112, 113, 127, 128, 129, 184, 185, 200, 257])
def test_sequence_edges(ctx, B, H, Hkv, hd, T):
    print(f"\n[attention split] B={B} H={H}/{Hkv} T={T} hd={hd}", flush=True)
    q, k, v = inputs(B, H, Hkv, T, hd, T)
    err = np.abs(attend(ctx, q, k, v) - reference(q, k, v)).max()
    print(f"  max|diff| {err:.3g}", flush=True)
    assert err <= 4e-5 * np.abs(v).max()


# (T 200 on the split kernel, 150 on the 16-row one)
@pytest.mark.parametrize("T", [150, 200])
@pytest.mark.parametrize("B,H,Hkv,hd", [(1, 4, 2, 128), (16, 16, 8, 64)])
def test_values_the_pieces_do_not_hold(ctx, B, H, Hkv, hd, T):
    print(f"\n[attention split] special values, hd={hd} T={T}", flush=True)
    q, k, v = inputs(B, H, Hkv, T, hd, 9)
    want = reference(q, k, v)
    # V around 2^-120: its low pieces would be subnormal
    small = np.float32(2.0**-120)
    got = attend(ctx, q, k, v * small).astype(np.float64) / float(small)
    assert np.abs(got - want).max() <= 4e-5 * np.abs(v).max()
    # queries of 2^100 beside keys of 2^-100
    got = attend(ctx, q * np.float32(2.0**100), k * np.float32(2.0**-100), v)
    assert np.abs(got - want).max() <= 4e-5 * np.abs(v).max()
    # an infinite value reaches the queries from its key on, in its column alone
    w = v.copy()
    w[:, :, 70, 3] = np.inf
    got = attend(ctx, q, k, w)
    assert np.all(got[:, :, 70:, 3] == np.inf)
    keep = np.ones(got.shape, bool)
    keep[:, :, 64:, 3] = False
    assert np.abs(got - want)[keep].max() <= 4e-5 * np.abs(v).max()
    # a NaN query row stays alone
    w = q.copy()
    w[:, :, 40, 0] = np.nan
    got = attend(ctx, w, k, v)
    assert np.all(np.isnan(got[:, :, 40]))
    keep = np.ones(T, bool)
    keep[40] = False
    assert np.abs(got - want)[:, :, keep].max() <= 4e-5 * np.abs(v).max()


@pytest.mark.parametrize("n", [1, 5, 40])
@pytest.mark.parametrize("B,H,Hkv,hd", [(1, 4, 2, 128), (16, 16, 8, 64)])
def test_leading_scores_of_minus_infinity(ctx, B, H, Hkv, hd, n):
    # the first n keys score -inf for the queries from n on, from an infinite
    # key and from a product that overflows: weight 0, as if they were masked
    T = 200
    print(f"\n[attention split] {n} leading scores of -inf, hd={hd}", flush=True)
    q, k, v = inputs(B, H, Hkv, T, hd, 11)
    q[..., 0], k[..., 0] = 0.0, 0.0
    want = reference(q[:, :, n:], k[:, :, n:], v[:, :, n:])
    bound = 4e-5 * np.abs(v).max()
    for big, low in ((np.float32(1.0), -np.float32(np.inf)), (np.float32(1e20), np.float32(-1e20))):
        w, x = q.copy(), k.copy()
        w[:, :, n:, 0], x[:, :, :n, 0] = big, low
        got = attend(ctx, w, x, v)
        assert np.abs(got[:, :, n:] - want).max() <= bound
    # (the overflowing product leaves the queries before n as they were)
    assert np.abs(got[:, :, :n] - reference(q[:, :, :n], k[:, :, :n], v[:, :, :n])).max() <= bound
    g = ctx.to_device(np.ones_like(q))
    grads = mh.causal_attention_backward(ctx, *(ctx.to_device(a) for a in (w, x, v)), g)
    assert all(np.isfinite(a.numpy()).all() for a in grads)
    # no score but -inf: NaN
    w[..., 0] = big
    assert np.isnan(attend(ctx, w, x, v)[:, :, :n]).all()


@pytest.mark.parametrize("B,H,Hkv,hd", [(1, 4, 2, 128), (16, 16, 8, 64)])
def test_small_probabilities_of_large_values(ctx, B, H, Hkv, hd):
    # key 0 has the whole weight and values of 0 in all columns but the first,
    # key 1 a probability of about 2^-n and values of about 2^e: outputs of
    # those columns are that product alone. Its relative error is the score's (n
    # in log2 units, rounded with its query's scale: 3 * 2^-24 n ln 2 < 2e-5) and
    # the product's
    T = 200
    print(f"\n[attention split] small probabilities, hd={hd}", flush=True)
    r = np.random.default_rng(3)
    for n, e in ((100, 90), (122, 110), (120, 20), (105, 124)):
        q, k, v = (np.zeros((B, h, T, hd), np.float32) for h in (H, Hkv, Hkv))
        q[..., 0] = r.uniform(1, 1.02, q.shape[:3])
        k[:, :, 1, 0] = -n * np.log(2) * np.sqrt(hd)
        k[:, :, 2:, 0] = -1e5
        v[:, :, 0, 0] = 1.0
        v[:, :, 1] = np.ldexp(r.uniform(1, 2, v[:, :, 1].shape), e)
        got, want = attend(ctx, q, k, v), reference(q, k, v)
        err = np.abs(got[:, :, 2:, 1:] / want[:, :, 2:, 1:] - 1).max()
        print(f"  2^-{n} of 2^{e}: max relative error {err:.3g}", flush=True)
        assert err <= 3e-5
