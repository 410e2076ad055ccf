"""Attention of many query positions over binary16 keys and values (attention_prompt.hip), by products of 16-bit parts: results are as near 64 bits as
over float32 caches, whatever the sizes of weights, values and features. Sizes at the edges of tiles (32
keys) and workgroups (64 or 128 rows), against 64 bits, the float32 cache and the kernel that takes a query row a workgroup."""
import numpy as np
import pytest

from mimir_amd import capi
from tests import test_gpu_decode_ops as T

pytestmark = pytest.mark.gpu


def both(q, k, v, scale, off):
    l = T.gpu.lib()
    got = T.attention(q, k, v, scale, causal=True, offset=off, kv_dt=capi.F16)
    assert T.last_kernel() == "attn_prompt_kernel"
    try:
        capi.check(l.mi355x_tune(b"attention.prompt", 0))
        return got, T.attention(q, k, v, scale, causal=True, offset=off, kv_dt=capi.F16)
    finally:
        capi.check(l.mi355x_tune(b"attention.prompt", 1))


def exact(q, k, v, scale, off):
    B, H, Q, D = q.shape
    g = H // k.shape[1]
    k64, v64 = (np.repeat(x.view(np.float16).astype(np.float64), g, axis=1) for x in (k, v))
    s = np.matmul(q.astype(np.float64) * scale, k64.transpose(0, 1, 3, 2))
    s[..., np.arange(k.shape[2])[None, :] > np.arange(Q)[:, None] + off] = -np.inf
    w = np.exp(s - s.max(-1, keepdims=True))
    return np.matmul(w, v64) / w.sum(-1, keepdims=True)


@pytest.mark.parametrize("B,H,HK,Q,K,D,spread", [
    (1, 4, 2, 64, 64, 128, 1),      # one step, one workgroup of two pairs
    (1, 4, 2, 65, 97, 64, 1),       # a row into the next workgroup; the last step's second tile holds one key
    (2, 4, 1, 96, 96, 128, 6),      # the last step is one tile: the second wavefront joins with fewer keys; scores far apart
    (1, 4, 4, 130, 159, 128, 0.01),  # ragged; weights all alike
    (4, 32, 8, 449, 70, 64, 1),     # workgroups of 128 rows; keys that end inside the third tile, most rows see all
])
def test_error_is_no_larger_than_with_float32_products(B, H, HK, Q, K, D, spread):
    rng = np.random.default_rng(Q + K)
    q = rng.normal(size=(B, H, Q, D)).astype(np.float32) * np.float32(spread)
    q *= np.exp(2 * rng.normal(size=(B, H, 1, D))).astype(np.float32) if spread == 1 else np.float32(1)  # features of unlike size
    k, v = (T.O.f32_to_f16(rng.normal(size=(B, HK, K, D)).astype(np.float32)) for _ in range(2))
    k, v = k.view(np.uint16), v.view(np.uint16)
    scale, off = 1 / np.sqrt(D), max(K - Q, 0)
    T.gpu.say(f"attention over binary16 B={B} H={H} Q={Q} K={K} D={D} spread={spread}")
    out, _ = T.attention(q, k, v, scale, causal=True, offset=off, kv_dt=capi.F16)
    assert T.last_kernel() == "attn_prompt_kernel"
    k32, v32 = (x.view(np.float16).astype(np.float32) for x in (k, v))
    single, _ = T.attention(q, k32, v32, scale, causal=True, offset=off, kv_dt=capi.F32)
    want = exact(q, k, v, scale, off)
    err, ref = (np.sqrt(np.mean((x.astype(np.float64) - want) ** 2)) for x in (out, single))
    # both are rounding errors of float32 sums of the same terms. The luck of the roundings may differ: a quarter, and one rounding of the results
    assert err <= 1.25 * ref + 2.0 ** -24 * np.sqrt(np.mean(want ** 2)), (err, ref)


@pytest.mark.parametrize("B,Q,D", [(1, 100, 128), (1, 100, 64), (4, 449, 64)])
def test_infinities_among_keys_and_queries(B, Q, D):
    """A NaN or an infinity in a key, a value or a row of Q gives every result the class (NaN, infinity, finite) that products of float32 give it."""
    rng = np.random.default_rng(Q)
    H, HK, K = 32 if B > 1 else 4, 2, 100
    q = rng.normal(size=(B, H, Q, D)).astype(np.float32)
    k = rng.normal(size=(B, HK, K, D)).astype(np.float32); v = rng.normal(size=(B, HK, K, D)).astype(np.float32)
    q[0, :, 40, 3] = 0.25; q[0, :, 40, 7] = 1e-20; q[0, :, 41, 7] = 0   # an exact binary16, one far below the row's largest, a zero
    k[0, 0, 20, 7] = np.inf      # scores of either infinity by the sign of q's feature 7
    k[0, 0, 50, 3] = -np.inf
    k[0, 1, 70, 2] = np.nan
    v[0, 1, 33, 5] = np.inf      # values seen whole from some row on and in part before
    v[0, 1, 34, 6] = -np.inf
    q[0, 0, 60, 9] = np.inf; q[0, 0, 60, 10] = 1e6
    k, v = T.O.f32_to_f16(k), T.O.f32_to_f16(v)
    T.gpu.say(f"attention over binary16, infinities, B={B} Q={Q} D={D}")
    (out, lse), (rows, lse_rows) = both(q, k, v, 1 / np.sqrt(D), 0)
    assert np.isnan(rows).any() and np.isfinite(rows).any()
    for got, want in ((out, rows), (lse, lse_rows)):
        fin = np.isfinite(want)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
        T.close(got[fin], want[fin])


def test_rows_that_see_no_key():
    """The first 40 rows see no key: zeros and -Inf."""
    rng = np.random.default_rng(3)
    q = rng.normal(size=(1, 4, 130, 128)).astype(np.float32)
    k, v = (T.O.f32_to_f16(rng.normal(size=(1, 2, 100, 128)).astype(np.float32)) for _ in range(2))
    T.gpu.say("attention over binary16, rows without keys")
    (out, lse), (rows, lse_rows) = both(q, k, v, 0.1, -40)
    assert not out[:, :, :40].any() and np.all(lse[:, :, :40] == -np.inf)
    T.close(out, rows); T.close(lse[:, :, 40:], lse_rows[:, :, 40:])


@pytest.mark.parametrize("D", [64, 128])
def test_small_weights_on_large_values(D):
    """The key of weight 1 has values of zero, the others of weights e^-8 down to e^-20 have large ones: every weight counts with its own 24 bits.
    Their relative error is the exponential's, a few 2^-24, and the argument's rounding, 20 x 2^-24: below 3e-6 in all."""
    rng = np.random.default_rng(5)
    q = np.zeros((1, 1, 64, D), np.float32); q[0, 0, :, 0] = np.linspace(8, 20, 64)
    k = np.zeros((1, 1, 64, D), np.float32); k[0, 0, 0, 0] = 1
    v = rng.normal(size=(1, 1, 64, D)).astype(np.float32) * 1000; v[0, 0, 0] = 0
    check_rows(q, k, v, 3e-6)


@pytest.mark.parametrize("D", [64, 128])
def test_small_features_of_q_by_large_keys(D):
    """Q's largest feature meets keys of zero, and one 2^-26 of it keys of 2^14: the scores (up to about 3) come from the small one,
    to float32's accuracy, and with them the weights: a few 2^-24 times 3."""
    rng = np.random.default_rng(6)
    q = rng.normal(size=(1, 1, 64, D)).astype(np.float32)
    q[..., 0] = 2.0 ** 11; q[..., 1] *= np.float32(2.0 ** -15)
    k = np.zeros((1, 1, 64, D), np.float32); k[..., 1] = rng.normal(size=64) * 2.0 ** 14
    check_rows(q, k, rng.normal(size=(1, 1, 64, D)).astype(np.float32), 2e-6)


def check_rows(q, k, v, bound):
    """Every row within `bound` of its root mean square of the same in 64 bits."""
    k, v = T.O.f32_to_f16(k).view(np.uint16), T.O.f32_to_f16(v).view(np.uint16)
    T.gpu.say(f"attention over binary16, unlike sizes, D={q.shape[3]}")
    got, _ = T.attention(q, k, v, 1.0, causal=False, kv_dt=capi.F16)
    assert T.last_kernel() == "attn_prompt_kernel"
    want = exact(q, k, v, 1.0, k.shape[2])  # an offset that hides no key
    err = max_row_error(got, want)
    assert err <= bound, err


def parts_of(q, scale, n):
    """Rows of Q as the sum of n binary16 each, the row's largest element in [2^14, 2^15) and each part 2^11 times what the ones ahead of it leave."""
    x = q * np.float32(scale)
    up = 2.0 ** (np.frexp(np.abs(x).max(-1, keepdims=True).astype(np.float64))[1] - 15)
    rest, held = x / up, 0
    for i in range(n):
        part = rest.astype(np.float16).astype(np.float64)
        held, rest = held + part * 2.0 ** (-11 * i), (rest - part) * 2048
    return held * up / scale


@pytest.mark.parametrize("B,H,Q,D,ratio,short", [
    (4, 32, 449, 128, 2.0 ** -27, 1), (4, 32, 449, 128, 2.0 ** -50, 3),   # workgroups of 128 rows
    (4, 32, 449, 128, 2.0 ** -120, 3),                                    # the largest is beyond 2^100: products of float32 operands
    (1, 4, 100, 128, 2.0 ** -36, 2), (1, 4, 100, 128, 2.0 ** -110, 3), (1, 4, 100, 128, 2.0 ** -120, 3), (1, 4, 100, 64, 2.0 ** -120, 3),  # workgroups of 64
])
def test_a_row_whose_features_lie_far_apart(B, H, Q, D, ratio, short):
    """One row of one sequence has a largest feature that meets keys of zero and one `ratio` of it whose products are scores of some units: that row and
    those that share its workgroup are within float32's rounding (scores up to about 8, weights to 8 x 2^-24, some 5e-7) of 64 bits, as all others are.
    With the row as `short` binary16 parts under one exponent it would be off by more than four times the bound."""
    rng = np.random.default_rng(Q + D)
    scale = np.float32(2.0 ** -27 / ratio)
    q = (rng.normal(size=(B, H, Q, D)) / np.sqrt(D) / scale).astype(np.float32); q[..., :2] = 0
    q[0, :, 70, 0] = 2.0 ** 13; q[0, :, 70, 1] = np.float32(1.2345678 * 2.0 ** 13 * ratio)
    k, v = (rng.normal(size=(B, 2, Q, D)).astype(np.float32) for _ in range(2))
    k[..., 0] = 0; k[..., 1] = np.clip(k[..., 1], -3, 3) * 2.0 ** 14
    k, v = T.O.f32_to_f16(k).view(np.uint16), T.O.f32_to_f16(v).view(np.uint16)
    want = exact(q, k, v, float(scale), 0)
    less = q[:1].astype(np.float64)
    less[0, :, 70] = parts_of(q[0, :, 70], scale, short)
    assert max_row_error(exact(less, k[:1], v[:1], float(scale), 0)[:, :, 70:71], want[:1, :, 70:71]) > 8e-6
    T.gpu.say(f"attention over binary16, features {ratio} apart, B={B} Q={Q} D={D}")
    got, _ = T.attention(q, k, v, float(scale), causal=True, offset=0, kv_dt=capi.F16)
    assert T.last_kernel() == "attn_prompt_kernel"
    err = max_row_error(got, want)
    assert err <= 2e-6, err


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("size", [2.0 ** -99, 2.0 ** -101, 2.0 ** -130])
def test_rows_of_next_to_nothing(size, D):
    """Rows of Q at and below the smallest that the parts hold: scores of nought to float32, so that all weights are one. The results' error is that of 65 added values."""
    rng = np.random.default_rng(D)
    q = (rng.normal(size=(1, 2, 64, D)) * size).astype(np.float32)
    k, v = (rng.normal(size=(1, 2, 65, D)).astype(np.float32) for _ in range(2))
    check_rows(q, k, v, 1e-6)


def max_row_error(got, want):
    return np.sqrt(np.mean((got.astype(np.float64) - want) ** 2, -1) / np.mean(want ** 2, -1)).max()


@pytest.mark.parametrize("B,H,Q,D", [(1, 2, 64, 128), (1, 2, 64, 64), (4, 32, 449, 128)])
def test_a_row_of_q_keeps_its_last_bits(B, H, Q, D):
    """Scores of some units that are the difference of two products 2^12 times as large, exact in float32: a feature of Q that lost the last of its 24 bits
    would move them by 2^-12. The results' error is the weights', a few 2^-24."""
    rng = np.random.default_rng(D)
    q = np.zeros((B, H, Q, D), np.float32)
    q[..., 0] = rng.uniform(1, 2, (B, H, Q)).astype(np.float32)
    q[..., 1] = q[..., 0].astype(np.float16)
    k = np.zeros((B, 1, Q, D), np.float32)
    k[..., 0] = rng.integers(-2, 3, (B, 1, Q)) * 4096.0; k[..., 1] = -k[..., 0]
    k, v = (T.O.f32_to_f16(x).view(np.uint16) for x in (k, rng.normal(size=(B, 1, Q, D)).astype(np.float32)))
    T.gpu.say(f"attention over binary16, last bits of Q, B={B} Q={Q} D={D}")
    got, _ = T.attention(q, k, v, 1.0, causal=False, kv_dt=capi.F16)
    assert T.last_kernel() == "attn_prompt_kernel"
    err = max_row_error(got, exact(q, k, v, 1.0, Q))
    assert err <= 1e-6, err


@pytest.mark.parametrize("D,K,low", [(64, 64, 75), (128, 64, 75), (128, 64, 86), (128, 100, 75)])
def test_weights_far_below_one(D, K, low):
    """The key of weight 1 has values of zero, the others' weights of e^-low down to e^-95 (below 2^-126, the smallest normal number, from e^-87.4 on) decide
    the results. Scores are exact: what remains is the exponential's error and the sums'. The first key is the last of the tiles that a wavefront takes, or the first,
    so that what came before it is scaled down by as much."""
    rng = np.random.default_rng(K)
    q = np.zeros((1, 1, 64, D), np.float32); q[..., 0] = 1
    v = (rng.uniform(0.5, 1, size=(1, 1, K, D)) * 60000).astype(np.float32)
    for at in (0, K - 1):
        k = np.zeros((1, 1, K, D), np.float32)
        k[0, 0, :, 0] = -np.round(rng.uniform(low, 95, K) * 16) / 16
        k[0, 0, at, 0] = 0
        w = v.copy(); w[0, 0, at] = 0
        check_rows(q, k, w, 1e-6)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("small", [2.0 ** -24, 2.0 ** -20])
def test_subnormal_keys_and_values(small, D):
    """All keys and values are subnormal binary16 numbers, down to the smallest. Scores of some units from all features: their rounding, 2^-24 of some 5, and that of their
    distance from the largest, 2^-24 of some 10, make some 1e-6 of the weights."""
    rng = np.random.default_rng(9)
    q = (rng.normal(size=(1, 2, 64, D)) / np.sqrt(D) / (8 * small)).astype(np.float32)
    k, v = (rng.integers(-15, 16, (1, 2, 64, D)).astype(np.float32) * np.float32(small) for _ in range(2))
    check_rows(q, k, v, 2e-6)
