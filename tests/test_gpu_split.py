"""The split-operand GEMMs (split_*: two fp16 values per operand value, three
products) forced onto shapes at the edges of their tiles, groups and panels:
exact integer products, the error against float64, operands of very different
scales, infinities, NaN and values outside the fp16 scaling's range, the fused
epilogues, and a call recorded into a HIP graph."""
import ctypes

import numpy as np
import pytest

import ncmhip
import oracle as O
from conftest import bits_equal, maxrel
from test_gpu_gpt2 import CASES as GPT2_CASES
from test_gpu_gpt2 import test_gpt2_grads as gpt2_step

pytestmark = pytest.mark.gpu
D = ncmhip.DeviceBuffer


@pytest.fixture(scope="module", autouse=True)
def device():
    ncmhip.init(0)
    ncmhip.load().arena_init(4 << 30)
    ncmhip.check()
    print("[gpu] split-operand GEMM tests on device 0", flush=True)


@pytest.fixture(params=[1064, 1128])
def tiles(request):
    lib = ncmhip.load()
    lib.ncm_hip_set_gemm_tiles(request.param)
    yield request.param
    lib.ncm_hip_set_gemm_tiles(0)


def run(x, W, dy, b=None, res=None, act="none", offset=0):
    """y, dx, dW, db of one layer (gradients into zeros); offset: floats by
    which every operand's address is moved off its 16-byte alignment."""
    M, K = x.shape
    N = W.shape[0]

    def put(a):
        buf = D.from_numpy(np.concatenate([np.zeros(offset, np.float32), a.reshape(-1)]))
        keep.append(buf)
        return buf.ptr + 4 * offset
    keep = []
    xp, Wp, dyp = put(x), put(W), put(dy)
    y = D.empty((M, N))
    g = [D.from_numpy(np.zeros(s, np.float32)) for s in ((M, K), (N, K), (N,))]
    ncmhip.linear_fwd(xp, Wp, None if b is None else D.from_numpy(b), y, M, N, K,
                      res=None if res is None else D.from_numpy(res), act=act)
    ncmhip.linear_bwd(xp, Wp, dyp, *g, M, N, K)
    return [y.numpy()] + [a.numpy() for a in g]


def exact(x, W, dy):
    x, W, dy = (a.astype(np.float64) for a in (x, W, dy))
    return x @ W.T, dy @ W, dy.T @ x, dy.sum(0)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("M,K,N", [(9, 1, 1), (63, 31, 65), (64, 128, 64), (65, 129, 127), (128, 260, 132),
                                   (129, 33, 129), (300, 513, 70), (1000, 96, 200)])
def test_exact_integer_products(tiles, M, K, N, offset):
    """x up to 2^13 needs both of its fp16 values; |sums| < 2^24, so y, dx, dW
    and db must equal the integer products bit for bit."""
    rng = np.random.default_rng(M + K + N)
    x = rng.integers(-5000, 5001, (M, K)).astype(np.float32)
    W, dy = (rng.integers(-2, 3, s).astype(np.float32) for s in ((N, K), (M, N)))
    for got, want in zip(run(x, W, dy, offset=offset), exact(x, W, dy)):
        assert np.abs(want).max() < 2 ** 24
        assert bits_equal(got.reshape(want.shape), want.astype(np.float32))


@pytest.mark.parametrize("M,K,N", [(64, 128, 192), (512, 896, 640), (1000, 1001, 515), (2048, 256, 128)])
def test_error_is_no_larger_than_the_fp32_kernels(tiles, M, K, N):
    """Relative 2-norm error against float64, and no element further off than
    the representation (2^-22 of each factor, 2^-22 for the dropped l.l) and
    one rounding per MFMA and group sum allow."""
    rng = np.random.default_rng(K)
    x, dy = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (M, N)))
    W = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    got = run(x, W, dy)
    ncmhip.load().ncm_hip_set_gemm_tiles(64)
    fp32 = run(x, W, dy)
    a = [np.abs(v).astype(np.float64) for v in (x, W, dy)]
    for g, f, want, size, red in zip(got, fp32, exact(x, W, dy), exact(*a), (K, N, M, M)):
        def err(v):
            return np.linalg.norm(v - want) / np.linalg.norm(want)
        assert err(g) <= 1.05 * err(f), (err(g), err(f))
        groups = -(-red // 128)
        assert np.all(np.abs(g - want) <= (3 * 2.0 ** -22 + (12 * min(groups, 1) + groups + 2) * 2.0 ** -23) * size)


def test_errors_cancel_over_rows_and_columns(tiles):
    """The 16-bit MFMAs round their sums one way; the operands' alternating
    signs turn half of the errors round, so means over many rows or columns of
    the output stay as close as single FP32 elements do (2.1e-7 .. 2.3e-7
    measured with the FP32 kernels, 8.6e-7 with every sign positive; the bar
    is the single element's error bound over sqrt(K) of random roundings)."""
    import math
    rng = np.random.default_rng(23)
    M, K, N = 1024, 2048, 768
    x, dy = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (M, N)))
    W = rng.standard_normal((N, K)).astype(np.float32)
    got, want = run(x, W, dy)[0], exact(x, W, dy)[0]
    bound = 2.0 ** -23 * math.sqrt(12)
    for axis in (0, 1):
        d = got.astype(np.float64).mean(axis) - want.mean(axis)
        assert np.linalg.norm(d) <= bound * np.linalg.norm(want.mean(axis))


def test_rows_and_groups_of_different_scales(tiles):
    """Every row, and every group of 128 k of a row, has its own exponent:
    operands scaled by powers of two from 2^-90 to 2^90 per row and group give
    the unscaled products' bits scaled, zero groups and rows included."""
    rng = np.random.default_rng(5)
    M, K, N = 70, 384, 66
    x, dy = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (M, N)))
    W = rng.standard_normal((N, K)).astype(np.float32)
    x[3] = 0.0
    x[5, 128:256] = 0.0
    base = run(x, W, dy)[0]
    ex, ew = rng.integers(-90, 91, (M, 1)), rng.integers(-30, 31, (N, 1))
    eg = np.repeat(rng.integers(-20, 21, 3), 128)[None]
    got = run(np.ldexp(x, ex + eg).astype(np.float32), np.ldexp(W, ew - eg).astype(np.float32), dy)[0]
    assert bits_equal(got, np.ldexp(base, ex + ew.T).astype(np.float32))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38, 1e-38, 1e-45])
def test_values_outside_the_scaling(tiles, value):
    """An infinity, a NaN, or a group whose largest value is beyond the scaling
    (its waves sum again in FP32): the same finite, infinite and NaN elements
    as float32 products, finite ones within the oracle's tolerance."""
    rng = np.random.default_rng(7)
    M, K, N = 130, 300, 140
    x, dy = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (M, N)))
    W = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    x[7, 40] = x[90, 299] = value
    W[20, 10] = value
    dy[50, 100] = value
    if abs(value) < 1:   # a whole row (of large values, every order of summing may overflow elsewhere)
        x[101] = np.float32(value) * np.sign(x[101])
    got = run(x, W, dy)
    with np.errstate(all="ignore"):
        want = [v.astype(np.float32) for v in exact(x, W, dy)]
    for g, w in zip(got, want):
        fine = np.isfinite(w)
        assert np.array_equal(np.isnan(g), np.isnan(w)) and np.array_equal(g[~fine & ~np.isnan(w)],
                                                                          w[~fine & ~np.isnan(w)])
        scale = np.abs(w[fine]) + (1.0 if abs(value) < 1e30 or not np.isfinite(value) else np.abs(w[fine]).max())
        assert np.all(np.abs(g[fine].astype(np.float64) - w[fine]) <= 1e-5 * scale)


def test_epilogues(tiles):
    rng = np.random.default_rng(11)
    M, K, N = 200, 256, 150
    x, dy, res = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (M, N), (M, N)))
    W, W2 = ((rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32) for _ in range(2))
    b = rng.standard_normal(N).astype(np.float32)
    y = O.linear_fwd(x, W, b)
    for act in ("none", "silu", "gelu", "gelu_tanh", "relu2"):
        want = y if act == "none" else np.maximum(y, 0) ** 2 if act == "relu2" else O.act(act, y)
        assert maxrel(run(x, W, dy, b, res, act)[0], want + res) <= 1e-5, act
    lib = ncmhip.load()
    xd, Wd, W2d, bd, rd, yd = (D.from_numpy(a) for a in (x, W, W2, b, res, res))
    ncmhip.linear_fwd(xd, Wd, bd, yd, M, N, K, res=yd)   # in place
    assert maxrel(yd.numpy(), y + res) <= 1e-5
    lib.linear_fwd_glu(xd.ptr, Wd.ptr, bd.ptr, rd.ptr, yd.ptr, M, N, K, 1)
    assert maxrel(yd.numpy(), O.act("silu", y) * res) <= 1e-5
    # the gated unit's own kernel needs its tiles to fill the CUs
    for m, n in ((M, N), (2100, 300)):
        xg = rng.standard_normal((m, K)).astype(np.float32)
        Wg, Wu = ((rng.standard_normal((n, K)) / np.sqrt(K)).astype(np.float32) for _ in range(2))
        bg = rng.standard_normal(n).astype(np.float32)
        o = D.empty((m, n))
        keep = [D.from_numpy(a) for a in (xg, Wg, bg, Wu)]
        lib.linear_fwd_gated(keep[0].ptr, keep[1].ptr, keep[2].ptr, keep[3].ptr, None, o.ptr, m, n, K, 1)
        ncmhip.check()
        assert maxrel(o.numpy(), O.act("silu", O.linear_fwd(xg, Wg, bg)) * O.linear_fwd(xg, Wu, None)) <= 1e-5


@pytest.mark.parametrize("case", range(min(2, len(GPT2_CASES))))
def test_training_step(tiles, case):
    """The tape's fused products (head-major q | k | v, pre-activation output,
    dX through the activation and into the heads) against the oracle."""
    gpt2_step(*GPT2_CASES[case])


def test_split_plans_sum_to_the_whole(tiles):
    """Few tiles and a long reduction: cut along k, partial tiles summed by the
    fixup; integers, so exact whatever the cut."""
    rng = np.random.default_rng(13)
    x = rng.integers(-3, 4, (40, 3000)).astype(np.float32)
    W, dy = rng.integers(-3, 4, (50, 3000)).astype(np.float32), rng.integers(-3, 4, (40, 50)).astype(np.float32)
    assert ncmhip.linear_route("fwd", 40, 50, 3000)[1] > 1
    for got, want in zip(run(x, W, dy), exact(x, W, dy)):
        assert bits_equal(got.reshape(want.shape), want.astype(np.float32))


def test_three_products_side_by_side(tiles):
    lib = ncmhip.load()
    rng = np.random.default_rng(17)
    M, K, ns = 200, 160, (192, 64, 40)
    x = rng.standard_normal((M, K)).astype(np.float32)
    Ws = [(rng.standard_normal((n, K)) / np.sqrt(K)).astype(np.float32) for n in ns]
    bs = [rng.standard_normal(n).astype(np.float32) if g != 1 else None for g, n in enumerate(ns)]
    xd, Wd = D.from_numpy(x), [D.from_numpy(W) for W in Ws]
    bd, yd = [None if b is None else D.from_numpy(b) for b in bs], [D.empty((M, n)) for n in ns]
    P3 = ctypes.c_void_p * 3
    fn = lib.ncm_linear_fwd3
    fn.restype, fn.argtypes = None, [ctypes.c_void_p, P3, P3, P3, ctypes.c_int * 3, ctypes.c_int64, ctypes.c_int]
    fn(xd.ptr, P3(*[w.ptr for w in Wd]), P3(*[None if b is None else b.ptr for b in bd]),
       P3(*[y.ptr for y in yd]), (ctypes.c_int * 3)(*ns), M, K)
    ncmhip.check()
    for y, W, b in zip(yd, Ws, bs):
        assert maxrel(y.numpy(), O.linear_fwd(x, W, b)) <= 1e-5


def test_capture_takes_the_fp32_kernel():
    """A captured call keeps no workspace address: it records the FP32 kernel,
    and replays on new inputs give that kernel's results."""
    M, N, K = 4096, 1024, 768
    assert ncmhip.linear_plan("fwd", M, N, K)[1] == 1   # no partial tiles, so no workspace at all
    assert ncmhip.linear_route("fwd", M, N, K)[0].startswith("split_")
    rng = np.random.default_rng(19)
    x, W, y = (D.from_numpy(rng.standard_normal(s).astype(np.float32)) for s in ((M, K), (N, K), (M, N)))
    ncmhip.linear_fwd(x, W, None, y, M, N, K)
    lib, hip = ncmhip.load(), ctypes.CDLL("libamdhip64.so")
    lib.ncm_hip_set_gemm_tiles(64)
    ncmhip.linear_fwd(x, W, None, y, M, N, K)
    lib.ncm_hip_set_gemm_tiles(0)
    ncmhip.sync()
    stream, graph, ex = ctypes.c_void_p(ncmhip.stream()), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 2) == 0
    ncmhip.linear_fwd(x, W, None, y, M, N, K)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        x.upload(rng.standard_normal((M, K)))
        assert hip.hipGraphLaunch(ex, stream) == 0
        got = y.numpy()
        lib.ncm_hip_set_gemm_tiles(64)
        ncmhip.linear_fwd(x, W, None, y, M, N, K)
        lib.ncm_hip_set_gemm_tiles(0)
        assert bits_equal(got, y.numpy())
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("mode", [64, 128, 1064, 1128])
@pytest.mark.parametrize("B,T,H,M", [(3, 64, 3, 128), (1, 128, 3, 68), (1, 192, 1, 64), (2, 64, 2, 256)])
def test_head_gradient_at_the_last_tiles(mode, B, T, H, M):
    """dX added into a head-major gradient where the outputs end inside a
    128 x 128 tile (an odd number of heads, an odd number of 64-row blocks):
    the waves past the end belong to no head and no sequence and must not touch
    memory; the guard floats around the gradient keep their bits."""
    rng = np.random.default_rng(29)
    lib, K, rows, guard = ncmhip.load(), 64 * H, B * T, 256
    dy, W = rng.integers(-3, 4, (rows, M)).astype(np.float32), rng.integers(-3, 4, (M, K)).astype(np.float32)
    old = rng.integers(-9, 10, (B, H, T, 64)).astype(np.float32)
    prod = (dy @ W).reshape(B, T, H, 64).transpose(0, 2, 1, 3)
    fn = lib.ncm_linear_bwd_heads
    vp, ci = ctypes.c_void_p, ctypes.c_int
    fn.restype, fn.argtypes = None, [vp, vp, vp, vp, ci, vp, vp, ci, ci, ci, ci]
    Wd, dyd = D.from_numpy(W), D.from_numpy(dy)
    print(f"[gpu] heads dX {B}x{T} x {H} heads, M {M}, mode {mode}", flush=True)
    lib.ncm_hip_set_gemm_tiles(mode)
    try:
        for beta in (0, 1):
            edge = np.full(guard, 7.5, np.float32)
            buf = D.from_numpy(np.concatenate([edge, old.reshape(-1), edge]))
            fn(None, Wd.ptr, dyd.ptr, buf.ptr + 4 * guard, beta, None, None, B, T, M, H)
            ncmhip.check()
            got = buf.numpy()
            assert bits_equal(got[:guard], edge) and bits_equal(got[-guard:], edge)
            assert bits_equal(got[guard:-guard].reshape(old.shape), old * beta + prod + np.float32(0.0))
    finally:
        lib.ncm_hip_set_gemm_tiles(0)


@pytest.mark.parametrize("M,N,K,offset", [(512, 4864, 896, 0), (2048, 1152, 896, 0), (600, 770, 515, 1)])
def test_capture_of_split_reductions(M, N, K, offset):
    """Calls whose FP32 plans cut the reduction (partial tiles in a workspace,
    bias sums in another): recorded right after the same calls ran eagerly on
    the split-operand kernels, and replayed on new inputs."""
    rng = np.random.default_rng(31)
    lib, hip = ncmhip.load(), ctypes.CDLL("libamdhip64.so")

    def put(shape):
        return D.from_numpy(np.zeros(int(np.prod(shape)) + offset, np.float32))

    def fill(buf, a):
        buf.upload(np.concatenate([np.zeros(offset, np.float32), a.reshape(-1)]))
    x, W, dy, y, dx, dW, db = (put(s) for s in ((M, K), (N, K), (M, N), (M, N), (M, K), (N, K), (N,)))
    p = [b.ptr + 4 * offset for b in (x, W, dy, y, dx, dW, db)]
    if offset == 0:
        assert ncmhip.linear_plan("fwd", M, N, K)[1] > 1
    assert ncmhip.linear_route("fwd", M, N, K)[0].startswith("split_")

    def step():
        ncmhip.linear_fwd(p[0], p[1], None, p[3], M, N, K)
        ncmhip.linear_bwd(p[0], p[1], p[2], p[4], p[5], p[6], M, N, K)
    step()
    ncmhip.sync()
    stream, graph, ex = ctypes.c_void_p(ncmhip.stream()), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 2) == 0
    step()
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        a = [rng.integers(-3, 4, s).astype(np.float32) for s in ((M, K), (N, K), (M, N))]
        for b, v in zip((x, W, dy), a):
            fill(b, v)
        for b, s in ((dx, (M, K)), (dW, (N, K)), (db, (N,))):
            fill(b, np.zeros(s, np.float32))
        assert hip.hipGraphLaunch(ex, stream) == 0
        for b, want in zip((y, dx, dW, db), exact(*a)):
            assert bits_equal(b.numpy()[offset:].reshape(want.shape), want.astype(np.float32))
        step()   # the eager calls between the replays
        ncmhip.sync()
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)


def _spread(rng, M, K, N, kind, e):
    """x, W, dy whose products are ordinary while values 2^e apart lie in one
    scale group of 128 (along the features for y and dx, the rows for dW)."""
    x, dy = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (M, N)))
    W = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    if kind == "units":       # features (and outputs, and rows) of different units, weights that make up for them
        f, o, r = (rng.integers(-e // 2, e // 2 + 1, (1, n)) for n in (K, N, M))
        x, W, dy = np.ldexp(x, f + r.T), np.ldexp(W, -f + o.T), np.ldexp(dy, -o - r.T)
    elif kind == "outlier":   # a large value where the other operand is zero
        x[:, 5::97] *= 2.0 ** e
        W[:, 5::97] = 0.0
        W[3::70] = 0.0
        dy[:, 3::70] *= 2.0 ** e
        x[7::90] = 0.0
        dy[7::90] *= 2.0 ** e
    elif kind == "reader":    # the same, but one output and one feature read the large value
        x[:, 5] *= 2.0 ** e
        W[:, 5] = 0.0
        W[-1, 5] = 1.0
        dy[4] *= 2.0 ** e
        x[4] = 0.0
        x[4, -1] = 1.0
    else:                     # tiny values beside ordinary ones, whole columns and rows of them
        x[:, ::3] *= 2.0 ** -e
        W[::3] *= 2.0 ** -e
        dy[1::3] *= 2.0 ** -e
        x[:, 1::3][rng.random(x[:, 1::3].shape) < 0.5] = 0.0
    return tuple(np.asarray(a, np.float32) for a in (x, W, dy))


@pytest.mark.parametrize("kind", ["units", "outlier", "reader", "tiny"])
@pytest.mark.parametrize("e", [14, 20, 24, 30, 40, 60])
@pytest.mark.parametrize("M,K,N", [(256, 384, 192), (131, 301, 141), (140, 100, 70)])
def test_values_far_apart_in_a_group(tiles, M, K, N, e, kind):
    """Two fp16 values hold a value to 2^-21 of itself down to 2^-19 of its
    group's largest: outputs that depend on smaller ones are summed again in
    FP32.  Element by element against sum |a b|, in float64: 2^-21 for each
    factor, 2^-22 for the dropped l.l, 2^-21 that may be lost before an output is
    summed again, and one rounding per MFMA and group sum."""
    x, W, dy = _spread(np.random.default_rng(37 + e), M, K, N, kind, e)
    got = run(x, W, dy)
    sizes = exact(*[np.abs(v) for v in (x, W, dy)])
    for g, want, size, red in zip(got, exact(x, W, dy), sizes, (K, N, M, M)):
        groups = -(-red // 128)
        bound = (7 * 2.0 ** -22 + (12 + groups + 2) * 2.0 ** -23) * size
        assert np.all(np.abs(g - want) <= bound), (np.max(np.abs(g - want) / (size + 1e-300)) * 2.0 ** 23, groups)


def test_units_of_features_in_every_form():
    """Features of different units through the default routes: q | k | v side
    by side, the gated unit and a cut reduction."""
    rng = np.random.default_rng(41)
    lib = ncmhip.load()
    M, K, ns = 520, 768, (192, 64, 128)
    f = rng.integers(-18, 19, (1, K))
    x = np.ldexp(rng.standard_normal((M, K)), f).astype(np.float32)
    Ws = [np.ldexp(rng.standard_normal((n, K)) / np.sqrt(K), -f).astype(np.float32) for n in ns]

    def close(got, x, W, slack=1.0):
        want, size = x.astype(np.float64) @ W.astype(np.float64).T, np.abs(x).astype(np.float64) @ np.abs(W).T
        assert np.all(np.abs(got - want) <= slack * (7 * 2.0 ** -22 + (12 + 6 + 2) * 2.0 ** -23) * size)
    xd, Wd, yd = D.from_numpy(x), [D.from_numpy(W) for W in Ws], [D.empty((M, n)) for n in ns]
    P3 = ctypes.c_void_p * 3
    fn = lib.ncm_linear_fwd3
    fn.restype, fn.argtypes = None, [ctypes.c_void_p, P3, P3, P3, ctypes.c_int * 3, ctypes.c_int64, ctypes.c_int]
    for mode in (1064, 1128):
        lib.ncm_hip_set_gemm_tiles(mode)
        fn(xd.ptr, P3(*[w.ptr for w in Wd]), P3(None, None, None), P3(*[y.ptr for y in yd]), (ctypes.c_int * 3)(*ns),
           M, K)
        ncmhip.check()
        for y, W in zip(yd, Ws):
            close(y.numpy(), x, W)
    n = 150   # the gated unit without an activation: the product of two sums, each within its bound
    Wg, Wu = (np.ldexp(rng.standard_normal((n, K)) / np.sqrt(K), -f).astype(np.float32) for _ in range(2))
    o, gd, ud = D.empty((M, n)), D.from_numpy(Wg), D.from_numpy(Wu)
    lib.linear_fwd_gated(xd.ptr, gd.ptr, None, ud.ptr, None, o.ptr, M, n, K, 0)
    ncmhip.check()
    lib.ncm_hip_set_gemm_tiles(0)
    a, b = (x.astype(np.float64) @ w.astype(np.float64).T for w in (Wg, Wu))
    sa, sb = (np.abs(x).astype(np.float64) @ np.abs(w).T for w in (Wg, Wu))
    c = 6 * 2.0 ** -22 + (12 + 6 + 2) * 2.0 ** -23
    assert np.all(np.abs(o.numpy() - a * b) <= c * (sa * np.abs(b) + sb * np.abs(a)) + c * c * sa * sb +
                  2.0 ** -23 * np.abs(a * b))
    xk, Wk = np.tile(x[:40], (1, 4)), np.tile(Ws[1], (1, 4))   # K = 3072, few tiles
    lib.ncm_hip_set_gemm_tiles(1064)
    assert ncmhip.linear_route("fwd", 40, 64, 3072)[1] > 1
    y = D.empty((40, 64))
    ncmhip.linear_fwd(D.from_numpy(xk), D.from_numpy(Wk), None, y, 40, 64, 3072)
    lib.ncm_hip_set_gemm_tiles(0)
    close(y.numpy(), xk, Wk, 2.0)
