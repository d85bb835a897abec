"""GPU checks of the split-bf16 attention backward (attention_bwd_split.hip:
heads of 64 and 128) against 64-bit softmax attention.

Bound, element by element, from sums of absolute values: a probability is off
by at most ~4e-5 of itself (its score and its log-sum-exp by 2e-5 each: 6*hd/16
roundings below 2^-23 of at most ~6 sqrt(hd) times the scale), dP and D by
6*hd/16 roundings of their absolute sums (3e-6), and the sums over the rows add
6*T/16 roundings (below 1e-5 here): together below 6e-5 of the same products
with absolute values everywhere.
"""
import numpy as np
import pytest

import midman_hip as mh

pytestmark = pytest.mark.gpu
REL = 6e-5


def reference(q, k, v, g, kv):
    """Gradients of batch element 0, kv head kv and its query heads, and their
    absolute-value sums."""
    _, H, T, hd = q.shape
    rep = H // k.shape[1]
    mask = np.tril(np.ones((T, T), bool))
    K, V = k[0, kv].astype(np.float64), v[0, kv].astype(np.float64)
    dq, dk, dv = np.empty((rep, T, hd)), np.zeros((T, hd)), np.zeros((T, hd))
    aq, ak, av = np.empty((rep, T, hd)), np.zeros((T, hd)), np.zeros((T, hd))
    for i in range(rep):
        Q, G = q[0, kv * rep + i].astype(np.float64), g[0, kv * rep + i].astype(np.float64)
        s = np.where(mask, Q @ K.T / np.sqrt(hd), -np.inf)
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        dp, ap = G @ V.T, np.abs(G) @ np.abs(V).T
        ds = p * (dp - (p * dp).sum(-1, keepdims=True)) / np.sqrt(hd)
        ad = p * (ap + (p * ap).sum(-1, keepdims=True)) / np.sqrt(hd)
        dq[i], aq[i] = ds @ K, ad @ np.abs(K)
        dk, ak = dk + ds.T @ Q, ak + ad.T @ np.abs(Q)
        dv, av = dv + p.T @ G, av + p.T @ np.abs(G)
    return (dq, dk, dv), (aq, ak, av)


def backward(ctx, q, k, v, g, kv):
    rep = q.shape[1] // k.shape[1]
    dq, dk, dv = mh.causal_attention_backward(ctx, *(ctx.to_device(x) for x in (q, k, v, g)))
    return dq.numpy()[0, kv * rep:(kv + 1) * rep], dk.numpy()[0, kv], dv.numpy()[0, kv]


def inputs(B, H, Hkv, T, hd, seed):
    r = np.random.default_rng(seed)
    f = lambda h: r.standard_normal((B, h, T, hd), dtype=np.float32)  # noqa: E731
    return f(H), f(Hkv), f(Hkv), f(H)


def check(got, want, bound, keep=(slice(None),) * 3):
    for name, a, w, b, s in zip(("dq", "dk", "dv"), got, want, bound, keep):
        sel = (slice(None), s) if name == "dq" else (s,)
        off = (np.abs(a - w) - REL * b)[sel].max()
        print(f"  {name} max|diff| {np.abs(a - w)[sel].max():.3g}", flush=True)
        assert off <= 0, (name, off)


# heads of 64 take these kernels from 200 positions and 256 blocks of 128 rows
# on, heads of 128 from 64 positions
@pytest.mark.parametrize("H,Hkv,hd,T", [(8, 4, 128, T) for T in (64, 65, 95, 96, 97, 127, 128, 129, 161, 257)]
                         + [(16, 8, 64, T) for T in (200, 223, 224, 225, 256, 257)]
                         + [(16, 16, 64, 289), (4, 4, 128, 289)])
def test_sequence_edges(ctx, H, Hkv, hd, T):
    print(f"\n[attention backward split] H={H}/{Hkv} T={T} hd={hd}", flush=True)
    a = inputs(8, H, Hkv, T, hd, T)
    want, bound = reference(*a, Hkv - 1)
    check(backward(ctx, *a, Hkv - 1), want, bound)


@pytest.mark.parametrize("H,Hkv,hd", [(8, 4, 128), (16, 8, 64), (16, 16, 64)])
def test_values_the_pieces_do_not_hold(ctx, H, Hkv, hd):
    T = 210
    print(f"\n[attention backward split] special values, hd={hd}", flush=True)
    q, k, v, g = inputs(8, H, Hkv, T, hd, 9)
    want, bound = reference(q, k, v, g, 1)
    # gradients around 2^-115 (their low pieces would be subnormal) and 2^90
    for e in (-115, 90):
        f = np.float32(2.0**e)
        got = backward(ctx, q, k, v, g * f, 1)
        check([x.astype(np.float64) / float(f) for x in got], want, bound)
    # queries of 2^100 beside keys of 2^-100: the same probabilities
    dq, dk, dv = backward(ctx, q * np.float32(2.0**100), k * np.float32(2.0**-100), v, g, 1)
    check([dq.astype(np.float64) * 2.0**100, dk.astype(np.float64) * 2.0**-100, dv], want, bound)
    # an infinite gradient stays in its query's dq and in the keys up to it
    w = g.copy()
    w[:, :, 140, 3] = np.inf
    got = backward(ctx, q, k, v, w, 1)
    assert not np.isfinite(got[0][:, 140]).any()
    assert np.all(got[2][:141, 3] == np.inf)
    others = np.arange(T) != 140
    check(got, want, bound, (others, slice(160, None), slice(160, None)))
    # a NaN query row: its own dq, and the keys it sees
    w = q.copy()
    w[:, :, 140, 0] = np.nan
    got = backward(ctx, w, k, v, g, 1)
    assert np.isnan(got[0][:, 140]).all() and np.isnan(got[2][:141]).all()
    check(got, want, bound, (others, slice(160, None), slice(160, None)))


@pytest.mark.parametrize("H,Hkv,hd", [(8, 8, 128), (16, 16, 64)])
def test_small_probabilities_of_large_gradients(ctx, H, Hkv, hd):
    # queries from 2 on give key 0 the whole weight (its values are 0) and key 1
    # a probability of about 2^-n: key 1's gradients are that probability alone
    # times one query's gradients of about 2^e. Relative error: the score's (n
    # in log2 units, a few roundings: 3 * 2^-24 n ln 2 < 2e-5) and the products'
    T = 210
    print(f"\n[attention backward split] small probabilities, hd={hd}", flush=True)
    r = np.random.default_rng(4)
    for n, e in ((100, 70), (122, 75), (122, 20), (105, 100)):
        q, k, v, g = (np.zeros((8, h, T, hd), np.float32) for h in (H, Hkv, Hkv, H))
        q[:, :, 2:, 0] = r.uniform(1, 1.02, q.shape[:2] + (T - 2,))
        k[:, :, 1, 0] = -n * np.log(2) * np.sqrt(hd)
        k[:, :, 2:, 0] = -1e5
        v[:, :, 1:] = r.uniform(1, 2, v[:, :, 1:].shape)
        g[:, :, 205] = np.ldexp(r.uniform(1, 2, g[:, :, 205].shape), e)
        dq, dk, dv = backward(ctx, q, k, v, g, 1)
        (wq, wk, wv), _ = reference(q, k, v, g, 1)
        err = [np.abs(a / w - 1).max() for a, w in ((dv[1], wv[1]), (dk[:2, 0], wk[:2, 0]),
                                                    (dq[:, 205, 0], wq[:, 205, 0]))]
        print(f"  2^-{n} of 2^{e}: max relative errors {err}", flush=True)
        assert max(err) <= 4e-5


@pytest.mark.parametrize("H,Hkv,hd", [(8, 8, 128), (16, 16, 64)])
def test_scores_beyond_the_lift(ctx, H, Hkv, hd):
    # all scores the same number of about -2^97: their f32 log-sum-exp is the
    # score itself, so every probability of the backward is 1
    T = 210
    print(f"\n[attention backward split] large scores, hd={hd}", flush=True)
    q, k, v, g = inputs(8, H, Hkv, T, hd, 5)
    q[...], k[...] = 0, 0
    q[..., 0], k[..., 0] = 2.0**50, -(2.0**50)
    _, _, dv = backward(ctx, q, k, v, g, 1)
    want = np.cumsum(g[0, 1, ::-1].astype(np.float64), 0)[::-1]
    size = np.cumsum(np.abs(g[0, 1, ::-1]).astype(np.float64), 0)[::-1]
    assert np.abs((dv - want) / size).max() <= REL
