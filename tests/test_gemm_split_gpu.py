"""The GEMM over split weights (csrc/gemm_split.hip, ops.split_weight / gemm_ws_f32_gpu) against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lk():
    import lokinfer_amd

    return lokinfer_amd


def G(lk, a):
    return lk.from_numpy(np.ascontiguousarray(a, np.float32), device="gpu", copy=True)


# (M, K, N): ragged rows, columns and K tails, K shorter than the wave groups, single rows and columns
SHAPES = [(1, 8, 1), (1, 16, 33), (31, 24, 32), (33, 40, 31), (59, 768, 2304), (200, 2048, 96), (487, 768, 768),
          (500, 72, 700), (487, 2056, 770), (1030, 136, 2100), (4100, 40, 2090), (8200, 256, 1056)]
# one per kernel of the launcher's rule: 32 x 32 with K over eight and four waves, 32 x 64 over four (steps of 16 and
# 32 k) and two wave groups, 32 x 128 over two and one, 64 x 128; the second half with one step or none for some of the
# groups
KERNELS = [(33, 776, 70), (31, 264, 2100), (487, 776, 768), (430, 2568, 700), (500, 136, 2304),
           (430, 264, 2300), (640, 48, 2990), (1500, 72, 2304), (32, 16, 2080), (600, 8, 768), (1000, 24, 700), (700, 40, 1300)]


@pytest.mark.parametrize("m,k,n", SHAPES + KERNELS)
def test_gemm_ws(lk, m, k, n):
    r = np.random.default_rng(m + 3 * k + 7 * n)
    a, w = r.standard_normal((m, k)).astype(np.float32), r.standard_normal((k, n)).astype(np.float32)
    ref, mag = a.astype(np.float64) @ w, np.abs(a).astype(np.float64) @ np.abs(w)
    bound = 2.0 ** -24 * (4 + np.sqrt(k)) * mag  # f32 sums of k products; random signs leave far less
    nn, nt = lk.ops.split_weight(G(lk, w)), lk.ops.split_weight(G(lk, w.T), nt=True)
    assert nn.shape == nt.shape == (k, n) and np.array_equal(nn.ws.numpy().view(np.uint8), nt.ws.numpy().view(np.uint8))
    y = lk.ops.gemm_ws_f32_gpu(G(lk, a), nn).numpy()
    assert y.shape == (m, n) and (np.abs(y - ref) <= bound).all()
    b, res = r.standard_normal(n).astype(np.float32), r.standard_normal((m, n)).astype(np.float32)
    z = lk.ops.gemm_ws_f32_gpu(G(lk, a), nn, G(lk, b), act="relu").numpy()
    assert (np.abs(z - np.maximum(ref + b, 0)) <= bound + 2.0 ** -23 * np.abs(ref + b)).all()
    z = lk.ops.gemm_ws_f32_gpu(G(lk, a), nn, G(lk, b), residual=G(lk, res)).numpy()
    assert (np.abs(z - (ref + b + res)) <= bound + 2.0 ** -22 * (np.abs(ref) + np.abs(b) + np.abs(res))).all()
    x = ref + b
    gelu = 0.5 * x * (1 + np.tanh(np.sqrt(2 / np.pi) * (x + 0.044715 * x ** 3)))
    z = lk.ops.gemm_ws_f32_gpu(G(lk, a), nn, G(lk, b), act="gelu").numpy()
    assert (np.abs(z - gelu) <= 1.2 * bound + 1e-6 * (1 + np.abs(x))).all()  # |gelu'| <= 1.13; f32 tanh


@pytest.mark.parametrize("m,k,n,planes", [s + (1,) for s in [(33, 40, 70), (200, 768, 64), (487, 768, 768), (8200, 64, 1056)] + KERNELS]
                         + [(59, 256, 96, 4), (256, 136, 768, 4)])
def test_gemm_ws_extreme_operands(lk, m, k, n, planes):
    """Infinities, NaN and values past the largest bf16 give what the f32 sum gives; rows of very different magnitude
    keep f32's relative error each; a weight holding such values too. Through every kernel, and the split-K planes."""
    r = np.random.default_rng(m + k + n)
    a = (r.standard_normal((m, k)) * 10.0 ** r.integers(-18, 18, (m, 1))).astype(np.float32)
    w = r.standard_normal((k, n)).astype(np.float32)
    y = _products(lk, a, w, planes)
    assert (np.abs(y - a.astype(np.float64) @ w) <= 2.0 ** -24 * (4 + np.sqrt(k)) * (np.abs(a).astype(np.float64) @ np.abs(w))).all()
    a = r.standard_normal((m, k)).astype(np.float32)
    for where in ("a", "w"):
        for bad in (np.inf, -np.inf, np.nan, 3.4e38):
            x, v = a.copy(), w.copy()
            if where == "a":
                x[m // 2, 3] = bad
            else:
                v[5, n - 1] = bad
                v[k - 1, 0] = bad
            with np.errstate(all="ignore"):
                ref = x.astype(np.float64) @ v
                bound = 2.0 ** -24 * (4 + np.sqrt(k)) * (np.abs(x).astype(np.float64) @ np.abs(v))  # f32 sums of k products
            got = _products(lk, x, v, planes)
            with np.errstate(all="ignore"):
                fits = np.abs(ref) < 3e38
                assert np.array_equal(np.isnan(ref), np.isnan(got))
                assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)].astype(np.float32))
                assert (np.abs(got[fits] - ref[fits]) <= bound[fits]).all()


@pytest.mark.parametrize("m,k,n,s", [(1, 64, 40, 3), (2, 16, 31, 5), (59, 2048, 768, 4), (320, 136, 700, 7), (400, 256, 768, 4),
                                     (32, 264, 700, 4), (100, 264, 768, 4), (256, 136, 768, 4), (300, 72, 760, 6)])
def test_gemm_ws_splitk(lk, m, k, n, s):
    r = np.random.default_rng(m + k)
    a, w = r.standard_normal((m, k)).astype(np.float32), r.standard_normal((k, n)).astype(np.float32)
    parts = lk.ops.gemm_ws_splitk_f32_gpu(G(lk, a), lk.ops.split_weight(G(lk, w)), s).numpy()
    assert parts.shape == (s, m, n)
    y = parts[:lk.ops.splitk_planes(m, n, s)].astype(np.float64).sum(0)
    bound = 2.0 ** -24 * (4 + np.sqrt(k)) * (np.abs(a).astype(np.float64) @ np.abs(w))  # f32 sums of k products
    assert (np.abs(y - a.astype(np.float64) @ w) <= bound).all()


def test_gemm_ws_refuses(lk):
    w = lk.ops.split_weight(G(lk, np.ones((12, 4))))
    with pytest.raises(ValueError):
        lk.ops.gemm_ws_f32_gpu(G(lk, np.ones((2, 12))), w)  # K % 8 != 0
    w = lk.ops.split_weight(G(lk, np.ones((16, 4))))
    with pytest.raises(ValueError):
        lk.ops.gemm_ws_f32_gpu(G(lk, np.ones((2, 8))), w)
    assert lk.ops.gemm_ws_f32_gpu(G(lk, np.ones((0, 16))), w).shape == (0, 4)


def _products(lk, a, w, planes):
    """a w, by one launch or as the sum of `planes` K ranges."""
    ws = lk.ops.split_weight(G(lk, w))
    if planes == 1:
        return lk.ops.gemm_ws_f32_gpu(G(lk, a), ws).numpy()
    with np.errstate(all="ignore"):
        return lk.ops.gemm_ws_splitk_f32_gpu(G(lk, a), ws, planes).numpy().sum(0)


@pytest.mark.parametrize("m,k,n,planes", [s + (1,) for s in KERNELS] + [(59, 256, 96, 4), (256, 136, 768, 4)])
def test_gemm_ws_largest_products(lk, m, k, n, planes):
    """A product that f32 holds is not lost where the operands' leading parts, both rounded up, multiply past it."""
    top = np.float32(0.9985 * 2.0 ** 64)
    a, w = np.zeros((m, k), np.float32), np.zeros((k, n), np.float32)
    want = np.zeros((m, n), np.float32)
    for i, (row, col, kk) in enumerate([(0, 0, 0), (m // 2, n // 3, k // 2), (m - 1, n - 1, k - 1)]):
        a[row, kk] = top * np.float32(2.0 ** (20 * i))
        w[kk, col] = top * np.float32(-2.0 ** (-20 * i))
        want[row, col] = a[row, kk] * w[kk, col]
    assert np.isfinite(want).all() and np.abs(want).max() > 3.39e38
    assert np.array_equal(_products(lk, a, w, planes), want)


@pytest.mark.parametrize("m,k,n,planes", [s + (1,) for s in KERNELS] + [(59, 256, 96, 4), (256, 136, 768, 4)])
@pytest.mark.parametrize("small", ["a", "w"])
def test_gemm_ws_small_operands(lk, m, k, n, planes, small):
    """Operands down to the smallest denormals, in rows of A or columns of W, enter with all their bits."""
    r = np.random.default_rng(m + k + n)
    a, w = r.standard_normal((m, k)) * 2.0 ** 60, r.standard_normal((k, n)) * 2.0 ** 60
    down = 2.0 ** -r.integers(160, 208, m if small == "a" else n)  # 2^-100 .. 2^-147
    a, w = (a * down[:, None], w) if small == "a" else (a, w * down)
    a, w = a.astype(np.float32), w.astype(np.float32)
    ref = a.astype(np.float64) @ w
    bound = 2.0 ** -24 * (4 + np.sqrt(k)) * (np.abs(a).astype(np.float64) @ np.abs(w))  # f32 sums of k products
    assert (np.abs(_products(lk, a, w, planes) - ref) <= bound).all()


def test_split_weight_parts(lk):
    """2^23 times every element is the sum of its parts down to the smallest denormals; only one that the factor takes past
    the largest float is stored whole behind a NaN (its columns leave the bf16 matrix cores)."""
    r = np.random.default_rng(9)
    w = (r.standard_normal((64, 96)) * 2.0 ** r.integers(-149, 125, (64, 96))).astype(np.float32)
    w[0, :8] = [0.0, -0.0, 2.0 ** -149, -(2.0 ** -110 - 2.0 ** -134), 3.4028235e38, 2.0 ** 105, np.inf, -(2.0 ** 105 - 2.0 ** 81)]
    p = lk.ops.split_weight(G(lk, w)).ws.numpy().view(np.uint16).reshape(3, 4, 3, 2, 32, 8).astype(np.uint32)
    p = p.transpose(2, 1, 3, 5, 0, 4).reshape(3, 64, 96)  # part, (chunk, half, k), (block, column)
    f = (p << 16).view(np.float32)
    whole = np.isnan(f[0])
    assert np.array_equal(whole, np.isfinite(w) & (np.abs(w) >= 2.0 ** 105))
    with np.errstate(invalid="ignore"):
        back = np.where(whole, (p[1] << 16 | p[2]).view(np.float32), ((f[0] + f[1]) + f[2]) * np.float32(2.0 ** -23))
    assert np.array_equal(back, w)


@pytest.mark.parametrize("m,k,n", KERNELS)
def test_gemm_ws_nan_weights(lk, m, k, n):
    """Every NaN stays one when a weight is laid out, also with all its significand bits in the low half."""
    r = np.random.default_rng(3)
    a, w = r.standard_normal((m, k)).astype(np.float32), r.standard_normal((k, n)).astype(np.float32)
    w.view(np.uint32)[1, 2], w.view(np.uint32)[k - 1, n - 1] = 0x7f800001, 0xff800001
    y = lk.ops.gemm_ws_f32_gpu(G(lk, a), lk.ops.split_weight(G(lk, w))).numpy()
    assert np.isnan(y[:, [2, n - 1]]).all() and np.isfinite(np.delete(y, [2, n - 1], 1)).all()


def test_weights_of_earlier_graphs(lk):
    """Kernels without the `scaled` attr (as saved graphs name them) lay out and read the parts of W itself: the same sums."""
    r = np.random.default_rng(4)
    m, k, n, s = 59, 256, 96, 4
    a, w, b = (G(lk, r.standard_normal(x)) for x in ((m, k), (k, n), (n,)))
    run, new = lk.ops._launch, lk.ops.split_weight(w)
    old = run("split_weight_f32_gpu", [w], [new.ws.shape], dict(nt=0))
    p = old.numpy().view(np.uint16).reshape(3, 16, 3, 2, 32, 8).astype(np.uint32).transpose(2, 1, 3, 5, 0, 4).reshape(3, k, n)
    f = (p << 16).view(np.float32)
    assert np.array_equal((f[0] + f[1]) + f[2], w.numpy())
    for name, args, out, attrs, want in [
            ("gemm_ws_f32_gpu", [a, old], (m, n), None, lk.ops.gemm_ws_f32_gpu(a, new)),
            ("gemm_ws_bias_gelu_f32_gpu", [a, old, b], (m, n), None, lk.ops.gemm_ws_f32_gpu(a, new, b, act="gelu")),
            ("gemm_ws_splitk_f32_gpu", [a, old], (s, m, n), dict(splits=s), lk.ops.gemm_ws_splitk_f32_gpu(a, new, s))]:
        assert np.array_equal(run(name, args, [out], attrs).numpy(), want.numpy())
