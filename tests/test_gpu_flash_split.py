"""The attention chains formed from bf16 parts (csrc/split_bf16.hpp, k_flash.hip) at their edges.

* Head dims and lengths around the tiles (32 tokens, 16-deep steps, dims padded to 32 or 64), forward
  and backward with the forward's score blocks kept, also for lengths that are no whole tiles, against
  float64. Bound: normwise 3e-6, about four times what float32 chains of this length show.
* Inputs past the scaled range (2^104), keys excluded by -inf in K: the float32 chains.
* Tiny gradients: no part is lost (the same bound). Score gradients past 2^104: float32 as well.
* Dot products past 2^80 that alpha brings back to ordinary scores.
* Factors alpha whose product with the scale is no normal number.
"""
import numpy as np
import pytest

import nnengine
from helpers import causal_mask, normal
from test_gpu_attn_chain import attn_mask, check, inputs, run

pytestmark = pytest.mark.gpu
TOL = 3e-6


def chain(e, q, k, v, g, mask, H, T, d, alpha, alpha2=1.0):
    q, k, v, g, mk = (e.tensor(x) for x in (q, k, v, g, mask))
    m = e.batched_matmul_reduce(q, k, H, "Max", True, False, alpha, True, mk)
    l = e.batched_matmul_softmax_denom(q, k, m, H, True, False, alpha, mk)
    vt = e.rearrange_3d(e.transpose(v), T, H, d)
    o = e.batched_matmul_softmax_apply(q, k, vt, m, l, H, True, False, alpha, mk)
    p = e.batched_matmul(g, v, H, True, False, alpha2)
    gt = e.rearrange_3d(e.transpose(g), T, H, d)
    dq, r = e.batched_matmul_softmax_backward_q(q, k, p, m, l, H, True, False, alpha, mk)
    dk, dv = e.batched_matmul_softmax_backward_kv(q, k, p, gt, r, m, l, H, True, False, alpha, mk)
    del p, gt, vt
    return [x.numpy() for x in (o, dq, dk, dv)]


def exact(q, k, v, g, mask, H, T, d, alpha, alpha2=1.0):
    q, k, v, g = (x.astype(np.float64).reshape(H, d, T) for x in (q, k, v, g))
    s = alpha * np.matmul(q.transpose(0, 2, 1), k) + mask.astype(np.float64)
    p = np.exp(s - s.max(axis=2, keepdims=True))
    p /= p.sum(axis=2, keepdims=True)
    o = np.matmul(p, v.transpose(0, 2, 1))
    dp = alpha2 * np.matmul(g.transpose(0, 2, 1), v)
    ds = p * (dp - (p * dp).sum(axis=2, keepdims=True)) * alpha
    dq = np.matmul(k, ds.transpose(0, 2, 1))
    return [o.reshape(H * T, d), dq.reshape(H * d, T), np.matmul(q, ds).reshape(H * d, T),
            np.matmul(g, p).reshape(H * d, T)]


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


@pytest.fixture(scope="module")
def no_blocks():
    """An engine that keeps no score blocks: the key-line pass forms the scores."""
    e = nnengine.Engine()
    e.set_score_budget(0)
    return e


@pytest.mark.parametrize("H,T,d", [(3, 32, 64), (2, 33, 64), (5, 100, 64), (2, 129, 40), (3, 500, 64), (2, 257, 16),
                                   (1, 64, 32), (4, 31, 20), (130, 70, 64), (2, 2050, 64),
                                   (2, 33, 68), (3, 100, 96), (2, 777, 128), (1, 32, 128), (5, 65, 124), (140, 40, 128)])
@pytest.mark.parametrize("masked", [False, True])
def test_edges(hip, H, T, d, masked):
    rng = np.random.default_rng(H * 31 + T + d)
    x = [normal(rng, (H * d, T)) for _ in range(4)]
    mask = causal_mask(T)
    if masked:   # general cells: finite values besides the excluded ones
        mask = mask + normal(rng, (T, T))
    got, ref = chain(hip, *x, mask, H, T, d, d ** -0.5), exact(*x, mask, H, T, d, d ** -0.5)
    for n, a, b in zip(("o", "dq", "dk", "dv"), got, ref):
        assert np.isfinite(a).all(), n
        assert rel(a, b) <= TOL, (n, rel(a, b))


@pytest.mark.parametrize("H,T,d", [(3, 100, 128), (2, 257, 96), (2, 70, 64), (2, 64, 32)])
@pytest.mark.parametrize("how", ["no_blocks", "no_output"])
def test_backward_without_the_forwards_work(hip, no_blocks, H, T, d, how):
    """Without score blocks (no budget for them) the key-line pass forms the scores; without the forward's output
    R comes from a pass over query lines."""
    rng = np.random.default_rng(T + d)
    x, mask, alpha = [normal(rng, (H * d, T)) for _ in range(4)], causal_mask(T), d ** -0.5
    ref = exact(*x, mask, H, T, d, alpha)
    if how == "no_blocks":
        got = chain(no_blocks, *x, mask, H, T, d, alpha)
    else:
        q, k, v, g, mk = (hip.tensor(a) for a in (*x, mask))
        m = hip.batched_matmul_reduce(q, k, H, "Max", True, False, alpha, True, mk)
        l = hip.batched_matmul_softmax_denom(q, k, m, H, True, False, alpha, mk)
        p = hip.batched_matmul(g, v, H, True, False)
        gt = hip.rearrange_3d(hip.transpose(g), T, H, d)
        dq, r = hip.batched_matmul_softmax_backward_q(q, k, p, m, l, H, True, False, alpha, mk)
        dk, dv = hip.batched_matmul_softmax_backward_kv(q, k, p, gt, r, m, l, H, True, False, alpha, mk)
        del p
        got, ref = [a.numpy() for a in (dq, dk, dv)], ref[1:]
    for a, b in zip(got, ref):
        assert rel(a, b) <= TOL


@pytest.mark.parametrize("B,H,T,dk", [(2, 2, 64, 128), (1, 3, 100, 96), (2, 1, 130, 72), (1, 2, 31, 128)])
@pytest.mark.parametrize("kind", ["alibi", "doc_alibi"])
def test_materialised_wide_heads(hip, cpu, B, H, T, dk, kind):
    """The materialised path (scores + mask, softmax rows, products) with heads wider than 64, against the oracle."""
    rng = np.random.default_rng(T + dk)
    doc = [np.cumsum(rng.random(T) < 0.04) for _ in range(B)] if kind == "doc_alibi" else None
    mask, arrs = attn_mask(B, H, T, doc_ids=doc), inputs(T, B * H, T, dk)
    for kw in (dict(), dict(order="kq"), dict(read_A=True)):
        check(run(hip, arrs, mask, B * H, T, dk ** -0.5, **kw), run(cpu, arrs, mask, B * H, T, dk ** -0.5, **kw))


@pytest.mark.parametrize("T,d", [(64, 64), (100, 32), (77, 64), (77, 128)])
def test_values_past_the_scaled_range(hip, T, d):
    """V of 1e33 (past 2^104) and Q of 1e32 against K of 1e-32, dO of 1e-30: the float32 chains."""
    rng = np.random.default_rng(T)
    H = 2
    q, k = normal(rng, (H * d, T)) * np.float32(1e32), normal(rng, (H * d, T)) * np.float32(1e-32)
    v, g = normal(rng, (H * d, T)) * np.float32(1e33), normal(rng, (H * d, T)) * np.float32(1e-30)
    got, ref = chain(hip, q, k, v, g, causal_mask(T), H, T, d, 0.125), exact(q, k, v, g, causal_mask(T), H, T, d, 0.125)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert rel(a, b) <= TOL


@pytest.mark.parametrize("T", [64, 77])
def test_minus_infinity_in_k(hip, T):
    H, d = 2, 64
    rng = np.random.default_rng(T)
    q, k, v, g = (normal(rng, (H * d, T)) for _ in range(4))
    q[5] = np.abs(q[5]) + 0.5
    k[5, 3] = -np.inf          # head 0, key 3: every score of it is -inf
    mask = causal_mask(T)
    kk, mm = k.copy(), np.repeat(mask[None], H, 0).copy()
    kk[5, 3] = 0.0
    mm[0, :, 3] = -np.inf
    mm[0, 3, 0] = 0.0          # (query 3 keeps other keys)
    o = chain(hip, q, k, v, g, mask, H, T, d, 0.125)[0]
    ref = exact(q, kk, v, g, mm, H, T, d, 0.125)[0]
    assert rel(o, ref) <= TOL


@pytest.mark.parametrize("scale", [1e-36, 1e-41])
def test_tiny_gradients(hip, scale):
    H, T, d = 3, 96, 64
    rng = np.random.default_rng(7)
    q, k, v = (normal(rng, (H * d, T)) for _ in range(3))
    g = (normal(rng, (H * d, T)).astype(np.float64) * scale).astype(np.float32)
    got, ref = chain(hip, q, k, v, g, causal_mask(T), H, T, d, 0.125), exact(q, k, v, g, causal_mask(T), H, T, d, 0.125)
    quantum = 2.0 ** -149 * np.sqrt(got[3].size)
    for a, b in zip(got[1:], ref[1:]):
        assert np.linalg.norm(a.astype(np.float64) - b) <= TOL * np.linalg.norm(b) + T * quantum


# lengths, head dims (32 and 64 wide tiles, one wave a SIMD at 128) and whether the forward keeps its score blocks
WIDTHS = [(64, 64, True), (77, 64, True), (96, 32, True), (70, 128, True), (100, 64, False), (64, 32, False)]


def chain_close(e, x, mask, H, T, d, alpha, alpha2=1.0):
    ref = exact(*x, mask, H, T, d, alpha, alpha2)
    assert all(np.abs(r).max() < 1e38 for r in ref)
    for n, a, b in zip(("o", "dq", "dk", "dv"), chain(e, *x, mask, H, T, d, alpha, alpha2), ref):
        assert np.isfinite(a).all(), n
        # (T sums of values that may round to multiples of 2^-149)
        assert np.linalg.norm(a - b) <= TOL * np.linalg.norm(b) + T * 2.0 ** -149 * np.sqrt(b.size), (n, rel(a, b))
    return ref


@pytest.mark.parametrize("T,d,keep", WIDTHS)
def test_score_gradients_past_the_scaled_range(hip, no_blocks, T, d, keep):
    """dO of 1e20 and V of 1e14: score gradients dS of 1e33 to 1e35, past 2^104, and finite products of them with Q
    and K of about 1."""
    rng = np.random.default_rng(T + d)
    H = 2
    q, k = normal(rng, (H * d, T)), normal(rng, (H * d, T))
    v, g = normal(rng, (H * d, T)) * np.float32(1e14), normal(rng, (H * d, T)) * np.float32(1e20)
    ref = chain_close(hip if keep else no_blocks, (q, k, v, g), causal_mask(T), H, T, d, d ** -0.5)
    assert np.abs(ref[1]).max() > 2.0 ** 108


@pytest.mark.parametrize("T,d,keep", WIDTHS)
@pytest.mark.parametrize("how", ["one_product", "cancelling", "negative_alpha"])
def test_scores_whose_scaled_sums_overflow(hip, no_blocks, T, d, keep, how):
    """Dot products below -2^80 (or with partial sums below it), infinite in the scaled sum, that alpha brings back
    to scores of about 1: such a key weighs as much as any other. Every row finds an ordinary score first."""
    rng = np.random.default_rng(T + d)
    H, alpha = 2, 2.0 ** -81
    q, k = np.zeros((H, d, T), np.float32), np.zeros((H, d, T), np.float32)
    q[:, 0] = 2.0 ** 50
    k[:, 0, 32:] = -(2.0 ** 31) * rng.uniform(0.75, 1.25, (H, T - 32))
    if how == "cancelling":   # (in two steps of 16 dims)
        q[:, 17], k[:, 17] = 2.0 ** 50, -0.375 * k[:, 0]
    if how == "negative_alpha":
        k, alpha = -k, -alpha
    x = q.reshape(H * d, T), k.reshape(H * d, T), normal(rng, (H * d, T)), normal(rng, (H * d, T))
    chain_close(hip if keep else no_blocks, x, causal_mask(T), H, T, d, alpha)


@pytest.mark.parametrize("T,d,keep", WIDTHS)
def test_small_factors(hip, no_blocks, T, d, keep):
    """alpha and the dP product's alpha below 2^-78: times the split's 2^-48 they are no normal numbers."""
    rng = np.random.default_rng(T + d)
    H, alpha, alpha2 = 2, float(np.float32(1.2345e-24)), float(np.float32(1.2345e-29))
    q, k = normal(rng, (H * d, T)) * np.float32(1e11), normal(rng, (H * d, T)) * np.float32(1e11)
    v, g = normal(rng, (H * d, T)), normal(rng, (H * d, T)) * np.float32(1e20)
    chain_close(hip if keep else no_blocks, (q, k, v, g), causal_mask(T), H, T, d, alpha, alpha2)


@pytest.mark.parametrize("T,d,keep", WIDTHS)
@pytest.mark.parametrize("big", ["q", "k", "v", "g"])
def test_large_values_within_the_scaled_range(hip, no_blocks, T, d, keep, big):
    """One operand spread over 2^87 to 2^103, just below the values whose parts overflow when scaled; its partner so
    small that scores (or dP) are of about 1, and V small enough that dK and dQ stay below 2^80. (O follows V and dV
    dO past it: the float32 chains of those.)"""
    rng = np.random.default_rng(T + d)
    H = 2
    x = {n: normal(rng, (H * d, T)) for n in "qkvg"}
    x[big] = (2.0 ** rng.uniform(87, 103, (H * d, T)) * rng.choice([-1.0, 1.0], (H * d, T))).astype(np.float32)
    x[{"q": "k", "k": "q", "v": "g", "g": "v"}[big]] *= np.float32(2.0 ** -103)
    if big in "qk":
        x["v"] *= np.float32(2.0 ** -40)
    chain_close(hip if keep else no_blocks, [x[n] for n in "qkvg"], causal_mask(T), H, T, d, d ** -0.5)
