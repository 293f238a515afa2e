"""Attention with head dimension 64 (operands split into fp16 pairs) at the
edges of its 64-query and 64-key tiles: the error against float64, operands of
very different scales, and inputs outside the range of the scaling, which take
the FP32 loop: infinities and NaN where exact arithmetic has them."""
import numpy as np
import pytest

import ncmhip

pytestmark = pytest.mark.gpu
D = ncmhip.DeviceBuffer


@pytest.fixture(scope="module", autouse=True)
def device():
    ncmhip.init(0)
    print("[gpu] split attention tests on device 0", flush=True)


def gpu(q, k, v, causal, mask=None):
    B, Hq, Tq, hd = q.shape
    Hkv, Tkv = k.shape[1:3]
    out = D.empty(q.shape)
    qd, kd, vd = D.from_numpy(q), D.from_numpy(k), D.from_numpy(v)
    if causal:
        ncmhip.call("sdpa_fwd_gqa_causal", qd, kd, vd, out, B, Hq, Hkv, Tq, Tkv, hd)
    else:
        ncmhip.call("sdpa_fwd_gqa", qd, kd, vd, None if mask is None else D.from_numpy(mask), out, B, Hq, Hkv, Tq,
                    Tkv, hd)
    return out.numpy()


def exact(q, k, v, causal, mask=None):
    q, k, v = (a.astype(np.float64) for a in (q, k, v))
    g = q.shape[1] // k.shape[1]
    k, v = np.repeat(k, g, 1), np.repeat(v, g, 1)
    with np.errstate(all="ignore"):
        s = q @ k.transpose(0, 1, 3, 2) / 8.0
        if mask is not None:
            s = s + mask
        if causal:
            Tq, Tkv = s.shape[2:]
            s[..., np.arange(Tkv)[None, :] > np.arange(Tq)[:, None] + Tkv - Tq] = -np.inf
        p = np.exp(s - s.max(-1, keepdims=True))
        return (p / p.sum(-1, keepdims=True)) @ v


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def data(rng, B, Hq, Hkv, Tq, Tkv):
    return [rng.standard_normal(s).astype(np.float32)
            for s in ((B, Hq, Tq, 64), (B, Hkv, Tkv, 64), (B, Hkv, Tkv, 64))]


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("B,Hq,Hkv,Tq,Tkv", [(1, 1, 1, 1, 1), (2, 4, 2, 17, 63), (1, 4, 1, 64, 64), (1, 2, 2, 65, 65),
                                             (3, 6, 2, 81, 81), (1, 2, 1, 127, 190), (1, 14, 2, 640, 700),
                                             (1, 2, 2, 1000, 1000)])
def test_shapes(B, Hq, Hkv, Tq, Tkv, causal):
    """h and l hold 22 bits, a dot product of 64 terms and the sums over keys
    round to 24: a few 2^-23 of the result's norm, 6e-7 = 5 x 2^-23."""
    q, k, v = data(np.random.default_rng(Tq + Tkv), B, Hq, Hkv, Tq, Tkv)
    print(f"[gpu] {B}x{Hq}/{Hkv} {Tq}x{Tkv} causal {causal}", flush=True)
    assert rel(gpu(q, k, v, causal), exact(q, k, v, causal)) < 6e-7


def test_scales():
    """Every query and column of V in its own power of two, dimensions up to
    2^14 apart (h and l hold 22 bits down to 2^-17 of a row's largest), and q
    and k beyond the range of the scaling (2^70: the FP32 loop)."""
    rng = np.random.default_rng(3)
    q, k, v = data(rng, 1, 2, 2, 130, 200)
    e = rng.integers(-7, 8, (1, 1, 1, 64))
    q, k = np.ldexp(q, e), np.ldexp(k, -e)
    q2, k2 = data(rng, 1, 2, 2, 130, 200)[:2]
    eq = rng.integers(-50, 3, (1, 2, 130, 1))
    ev = rng.integers(-50, 50, (1, 2, 1, 64))
    for a, b, c in ((q, k, v), (np.ldexp(q2, eq), k2, v), (q2, k2, np.ldexp(v, ev)),
                    (q2 * 2.0 ** 55, k2 * 2.0 ** -55, v), (q2 * 2.0 ** 70, k2 * 2.0 ** -70, v)):
        a, b, c = (np.asarray(t, np.float32) for t in (a, b, c))
        got, want = gpu(a, b, c, 0), exact(a, b, c, 0)
        assert all(rel(got[..., d], want[..., d]) < 1.2e-6 for d in range(64))   # 10 x 2^-23 of each column


def test_nonfinite():
    rng = np.random.default_rng(5)
    q, k, v = data(rng, 1, 2, 1, 100, 150)
    mask = np.where(rng.random((100, 150)) < 0.3, -np.inf, 0.0).astype(np.float32)
    mask[:, 0] = 0.0
    assert rel(gpu(q, k, v, 0, mask), exact(q, k, v, 0, mask)) < 6e-7
    low = np.where(np.isinf(mask), np.finfo(np.float32).min, 0.0).astype(np.float32)
    assert rel(gpu(q, k, v, 0, low), exact(q, k, v, 0, low)) < 6e-7
    k1, v1, v2, q1 = k.copy(), v.copy(), v.copy(), np.abs(q)
    k1[0, 0, 70, 5] = -np.inf          # scores of -inf: the key takes no part
    v1[0, 0, 149, 7] = np.inf
    v2[0, 0, 3, 9] = np.nan
    for a, b, c in ((q1, k1, v), (q, k, v1), (q, k, v2)):
        got, want = gpu(a, b, c, 0), exact(a, b, c, 0)
        fin = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), fin) and np.array_equal(np.isnan(got), np.isnan(want))
        assert rel(got[fin], want[fin]) < 1e-6


def close(got, want, q, k, v, causal, mask=None):
    """Element by element, in float64, against sum p |v| / sum p: a score is off
    by sum |q k| / 8 times the 2^-21 of its pairs' representation (2 x 2^-23, l.l
    2^-22) and some ten roundings of the sums (10 x 2^-24), and by 2^-23 of the
    larger of 1 and the scores that the bound lets pass; p and V by as much of
    themselves, their sum by 2^-21 and its roundings, one a tile."""
    size = exact(q, k, np.abs(v), causal, mask)
    g = q.shape[1] // k.shape[1]
    s = np.abs(q.astype(np.float64)) @ np.repeat(np.abs(k.astype(np.float64)), g, 1).transpose(0, 1, 3, 2) / 8.0
    if causal:
        Tq, Tkv = s.shape[2:]
        s[..., np.arange(Tkv)[None, :] > np.arange(Tq)[:, None] + Tkv - Tq] = 0.0
    scores = s.max(-1, keepdims=True) * (2.0 ** -21 + 10 * 2.0 ** -24) + 2.0 ** -23
    rel = 2.0 ** -21 + 2.0 ** -21 + (k.shape[2] // 64 + 12) * 2.0 ** -23
    return np.all(np.abs(got - want) <= (2 * scores + rel) * size)


@pytest.mark.parametrize("big", [1e6, 1e9, 1e12, 1e15, -1e17])
@pytest.mark.parametrize("causal", [0, 1])
def test_large_values_at_keys_that_do_not_count(causal, big):
    """Keys that the mask removes, keys to come, and keys whose softmax weight is
    nothing, with a V that is 10^6 .. 10^17 times the others': the outputs are
    those of the keys that count."""
    rng = np.random.default_rng(11)
    q, k, v = data(rng, 2, 4, 2, 130, 200)
    mask = np.zeros((130, 200), np.float32)
    if causal:
        v[:, :, 199] *= big            # seen by the last query only
        v[0, :, 150, ::3] = big        # by some fifty of them
        want = exact(q, k, v, 1)
        got = gpu(q, k, v, 1)
    else:
        for fill in (-np.inf, np.finfo(np.float32).min, -1e30):
            mask[:, 5] = mask[:, 70:72] = mask[3:, 199] = fill
            v[:, :, 5] = v[:, :, 70:72] = big
            v[0, :, 199, 1::2] = big
            want, got = exact(q, k, v, 0, mask), gpu(q, k, v, 0, mask)
            assert close(got, want, q, k, v, 0, mask)
        # not masked: a score some 25 below the others', so 10^-11 of the weight
        q[..., 0] = 40.0
        k[..., 0] = 0.0
        k[:, :, 33, 0] = -5.0
        mask = None
        v[:, :, 33] = big
        want, got = exact(q, k, v, 0), gpu(q, k, v, 0)
    assert close(got, want, q, k, v, causal, mask)


@pytest.mark.parametrize("e", [8, 14, 20, 30])
@pytest.mark.parametrize("Tq,Tkv", [(130, 200), (700, 700)])
def test_units_of_dimensions(Tq, Tkv, e):
    """Dimensions of q in units up to 2^e apart, those of k in the inverse ones;
    columns of V with values 2^2e apart."""
    rng = np.random.default_rng(13 + e)
    q, k, v = data(rng, 1, 2, 1, Tq, Tkv)
    f = rng.integers(-e, e + 1, (1, 1, 1, 64))
    q, k = np.ldexp(q, f).astype(np.float32), np.ldexp(k, -f).astype(np.float32)
    v = np.ldexp(v, rng.integers(-e, e + 1, v.shape)).astype(np.float32)
    for causal in (0, 1):
        assert close(gpu(q, k, v, causal), exact(q, k, v, causal), q, k, v, causal)


def test_peaked_softmax():
    """Scores of a wide range (weights from 1 down to nothing), queries and rows
    of zeros, zero columns of V."""
    rng = np.random.default_rng(17)
    q, k, v = data(rng, 1, 2, 2, 300, 400)
    q *= 12.0
    q[0, 0, 7] = k[0, 1, 9] = 0.0
    v[..., 5] = 0.0
    v[0, 0, 100:, 6] = 0.0
    for causal in (0, 1):
        assert close(gpu(q, k, v, causal), exact(q, k, v, causal), q, k, v, causal)
