"""Winograd conv family on the GPU (wino_tf* -> wino_mm* -> wino_adain_affine) vs the float64 direct conv of the
oracle, over the reference's test shapes (tests/kernels/test_winograd_gpu.py:40-175 in lariaus/lokinfer) plus the
Kokoro generator's: conv 1e-4, snake / leaky fused 2e-4, stats mean 1e-5 and inverse std 1e-4."""
import math

import numpy as np
import pytest

from lokinfer_amd import winograd as W
from oracle import kernels as K

pytestmark = pytest.mark.gpu


def G(lk, a):
    return lk.from_numpy(np.ascontiguousarray(a, np.float32), device="gpu", copy=True)


def close(got, ref, tol):
    got = got.numpy() if hasattr(got, "numpy") else np.asarray(got)
    ref = np.asarray(ref, np.float64)
    assert got.shape == ref.shape, (got.shape, ref.shape)
    err = np.abs(got.astype(np.float64) - ref)
    bound = tol + tol * np.abs(ref)
    assert (err <= bound).all(), f"max excess {np.max(err - bound):.3e}"


def _pad(k, d):
    return d * (k // 2) if k % 2 == 0 else d * (k - 1) // 2


def _case(seed, l, ci, co, k):
    r = np.random.default_rng(seed)
    x = r.standard_normal((l, ci)).astype(np.float32)
    w = (r.standard_normal((co, ci, k)) / math.sqrt(ci * k)).astype(np.float32)
    b = r.standard_normal(co).astype(np.float32)
    return r, x, w, b


def _direct(h, w, b, pad, d, res=None, scale=1.0):
    # oracle conv takes w [Co, K, Ci]
    return K.conv1d_lc(h, np.transpose(w, (0, 2, 1)), b, padding=pad, dilation=d, residual=res, out_scale=scale)


CONVS = [(128, 128, 1000, 11, 5), (128, 128, 777, 7, 3), (256, 256, 300, 3, 1), (128, 128, 1001, 3, 5),
         (256, 256, 513, 7, 1), (128, 128, 37, 11, 3), (16, 64, 5, 3, 1), (128, 64, 1001, 7, 1),
         (32, 128, 70, 5, 2), (64, 64, 9, 12, 1), (16, 64, 40, 4, 1), (128, 128, 2, 3, 1),
         (256, 256, 1770, 3, 3), (128, 128, 10621, 11, 5),
         # one tap group with 48- and 32-channel pipeline steps (Ci / 16 divisible by 3, by 2)
         (144, 64, 500, 3, 1), (48, 128, 301, 3, 2), (96, 64, 257, 3, 1)]


@pytest.mark.parametrize("ci,co,l,k,d", CONVS)
@pytest.mark.parametrize("res", [False, True])
def test_wino_conv1d(gpu, ci, co, l, k, d, res):
    lk = gpu
    r, x, w, b = _case(ci + l + k + d, l, ci, co, k)
    pad = _pad(k, d)
    u, tr = W.wino_weights(w)
    if res:
        rr = r.standard_normal((l + 2 * pad - d * (k - 1), co)).astype(np.float32)
        ref = _direct(x, w, b, pad, d, rr, 0.5)
        got = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), k, residual=G(lk, rr),
                                            out_scale=0.5, padding=pad, dilation=d)
    else:
        ref = _direct(x, w, b, pad, d)
        got = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), k, padding=pad, dilation=d)
    close(got, ref, 1e-4)


def _affine(r, ci):
    return np.stack([r.standard_normal(ci) * 0.5, r.uniform(0.5, 1.5, ci), r.standard_normal(ci) * 0.3]).astype(
        np.float32)


@pytest.mark.parametrize("ci,co,l,k,d", [(128, 128, 1000, 11, 5), (256, 256, 300, 3, 3), (128, 128, 501, 7, 1)])
def test_wino_conv1d_snake(gpu, ci, co, l, k, d):
    lk = gpu
    r, x, w, b = _case(l + k, l, ci, co, k)
    x = x * 2
    af, alpha = _affine(r, ci), r.uniform(0.2, 3.0, ci).astype(np.float32)
    pad = _pad(k, d)
    ref = _direct(K.affine_act(x, af, alpha, "snake"), w, b, pad, d)
    u, tr = W.wino_weights(w)
    got = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), k, padding=pad, dilation=d,
                                        affine=G(lk, af), alpha=G(lk, alpha))
    close(got, ref, 2e-4)


@pytest.mark.parametrize("ci,co,l", [(1104, 1024, 147), (528, 1024, 60), (256, 256, 294)])
@pytest.mark.parametrize("res", [False, True])
def test_wino_conv1d_leaky(gpu, ci, co, l, res):
    lk = gpu
    r, x, w, b = _case(l + ci, l, ci, co, 3)
    x = x * 2
    af = _affine(r, ci)
    h = K.affine_act(x, af, None, "leaky", 0.2)
    u, tr = W.wino_weights(w)
    kw, rr = {}, None
    if res:
        rr = r.standard_normal((l, co)).astype(np.float32)
        kw = dict(residual=G(lk, rr), out_scale=0.7071)
    ref = _direct(h, w, b, 1, 1, rr, 0.7071 if res else 1.0)
    got = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), 3, padding=1, affine=G(lk, af),
                                        slope=0.2, **kw)
    close(got, ref, 2e-4)


def _check_affine(af, y, gb, co):
    y64 = y.astype(np.float64)
    mean, var = y64.mean(0), y64.var(0)
    np.testing.assert_allclose(af[0], mean, atol=1e-5, rtol=1e-5)
    np.testing.assert_allclose(af[1], (1 + gb[:co]) / np.sqrt(var + 1e-5), rtol=1e-4)
    assert np.array_equal(af[2], gb[co:])


@pytest.mark.parametrize("ci,co,l,k,d", [(128, 128, 1000, 11, 5), (128, 128, 777, 7, 3), (256, 256, 300, 3, 1),
                                         (128, 128, 129, 3, 1), (128, 64, 5, 7, 3), (64, 64, 300, 12, 2),
                                         (256, 256, 700, 7, 3), (256, 128, 300, 11, 5)])  # split-K, dilated stats
@pytest.mark.parametrize("res", [False, True])
def test_wino_stats_epilogue_affine(gpu, ci, co, l, k, d, res):
    lk = gpu
    r, x, w, b = _case(l + k + d, l, ci, co, k)
    b = b + 3  # a non-zero mean
    gb = (r.standard_normal(2 * co) * 0.3).astype(np.float32)
    pad = _pad(k, d)
    lo = l + 2 * pad - d * (k - 1)  # even K: one row longer per dilation
    u, tr = W.wino_weights(w)
    kw, rr = {}, None
    if res:
        rr = r.standard_normal((lo, co)).astype(np.float32)
        kw = dict(residual=G(lk, rr), out_scale=0.5)
    y, st = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), k, padding=pad, dilation=d,
                                          stats=True, **kw)
    assert st.shape == (W.stats_chunks(lo, d) * d, co, 2)
    close(y, _direct(x, w, b, pad, d, rr, 0.5 if res else 1.0), 1e-4)
    yn = y.numpy()
    if d == 1:  # the statistics layout equals channel_stats_lc's for d = 1
        np.testing.assert_allclose(st.numpy(), K.channel_stats_lc(yn), rtol=1e-4, atol=1e-4)
    af = lk.ops.wino_adain_affine_lc_f32_gpu(st, G(lk, gb), lo, dilation=d).numpy()
    _check_affine(af, yn, gb, co)


def test_wino_affine_padded_channels(gpu):
    """Creal < C: channels past Creal get an all-zero affine (the decoder's padded widths)."""
    lk = gpu
    r, x, w, b = _case(5, 300, 128, 128, 3)
    u, tr = W.wino_weights(w)
    y, st = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), 3, padding=1, stats=True)
    gb = (r.standard_normal(2 * 100) * 0.3).astype(np.float32)
    af = lk.ops.wino_adain_affine_lc_f32_gpu(st, G(lk, gb), 300).numpy()
    assert not af[:, 100:].any()
    y64 = y.numpy().astype(np.float64)[:, :100]
    np.testing.assert_allclose(af[0, :100], y64.mean(0), atol=1e-5, rtol=1e-5)
    np.testing.assert_allclose(af[1, :100], (1 + gb[:100]) / np.sqrt(y64.var(0) + 1e-5), rtol=1e-4)
    assert np.array_equal(af[2, :100], gb[100:])


@pytest.mark.parametrize("ci,co,l,d", [(256, 256, 300, 1), (128, 128, 1001, 5), (16, 64, 5, 1), (128, 128, 4097, 3)])
@pytest.mark.parametrize("stats", [False, True])
def test_wino_f23(gpu, ci, co, l, d, stats):
    lk = gpu
    r, x, w, b = _case(ci + l + d, l, ci, co, 3)
    rr = r.standard_normal((l, co)).astype(np.float32)
    ref = _direct(x, w, b, d, d, rr, 0.5)
    u, tr = W.wino_weights(w, tile=2)
    assert u.shape[0] == 4
    out = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), 3, residual=G(lk, rr), out_scale=0.5,
                                        padding=d, dilation=d, stats=stats)
    if stats:
        out, st = out
        af = lk.ops.wino_adain_affine_lc_f32_gpu(st, G(lk, np.zeros(2 * co, np.float32)), l, dilation=d).numpy()
        np.testing.assert_allclose(af[0], out.numpy().astype(np.float64).mean(0), atol=1e-5, rtol=1e-5)
    close(out, ref, 1e-4)


def test_wino_split_ops_and_rejects(gpu):
    """The two-launch pair called op by op equals conv1d_wino; bad operands raise before any launch."""
    lk = gpu
    r, x, w, b = _case(11, 200, 64, 64, 7)
    u, tr = W.wino_weights(w)
    attrs = dict(dilation=3, groups=2, kernel=7, padding=9, tile=4)
    v = lk.ops.wino_tf_lc_f32_gpu(G(lk, x), G(lk, tr), **attrs)
    assert v.shape == (W.tiles_rows(200, 3, 2, 4, 7), 64)
    y = lk.ops.wino_mm_lc_f32_gpu(v, G(lk, u), G(lk, b), G(lk, tr), G(lk, x), **attrs)
    y2 = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), 7, padding=9, dilation=3)
    assert np.array_equal(y.numpy(), y2.numpy())
    with pytest.raises(ValueError):  # Ci not a multiple of 16
        lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x[:, :40]), G(lk, u), G(lk, b), G(lk, tr), 7, padding=9, dilation=3)
    with pytest.raises(ValueError):  # padding not a multiple of the dilation
        lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), 7, padding=8, dilation=3)
    with pytest.raises(ValueError):  # U for another kernel size
        lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), 3, padding=3, dilation=3)


def _mm_workgroups(lo, co, d, tile):
    """Workgroups of one wino_mm launch (csrc/winograd.hip lk_hip_wino_mm_lc_f32, no split): 64 output channels x
    64 tiles of one residue class each. Above 512 (two per CU) the three-per-CU instantiations run."""
    tiles = -(-(-(-lo // d)) // tile)
    return (co // 64) * (-(-tiles // 64)) * d


# Grids above 512 workgroups: the only shapes that select winoMmKernel<4,6,1,3>, <4,7,2,3> and <4,7,3,3> (the
# Kokoro-487 generator's convs). Each runs with the fused affine + Snake, the residual and the stats epilogue,
# as the generator's resblocks do.
LARGE = [(128, 128, 80000, 11, 5), (256, 256, 48880, 7, 3), (128, 128, 70000, 3, 1), (128, 128, 80000, 3, 5)]


@pytest.mark.parametrize("ci,co,l,k,d", LARGE)
def test_wino_large_grid_instantiations(gpu, ci, co, l, k, d):
    lk = gpu
    r, x, w, b = _case(l + 3 * k + d, l, ci, co, k)
    pad = _pad(k, d)
    assert _mm_workgroups(l, co, d, 4) > 512
    af, alpha = _affine(r, ci), r.uniform(0.2, 3.0, ci).astype(np.float32)
    rr = r.standard_normal((l, co)).astype(np.float32)
    u, tr = W.wino_weights(w)
    y, st = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), k, residual=G(lk, rr),
                                          padding=pad, dilation=d, affine=G(lk, af), alpha=G(lk, alpha), stats=True)
    ref = _direct(K.affine_act(x, af, alpha, "snake"), w, b, pad, d, rr)
    close(y, ref, 2e-4)
    yn = y.numpy()
    assert st.shape == (W.stats_chunks(l, d) * d, co, 2)
    if d == 1:
        np.testing.assert_allclose(st.numpy(), K.channel_stats_lc(yn), rtol=1e-4, atol=1e-4)
    gb = (r.standard_normal(2 * co) * 0.3).astype(np.float32)
    af2 = lk.ops.wino_adain_affine_lc_f32_gpu(st, G(lk, gb), l, dilation=d).numpy()
    _check_affine(af2, yn, gb, co)


@pytest.mark.parametrize("ci,co,l,k,d", CONVS[:10] + [(1104, 1024, 300, 3, 1), (144, 64, 500, 3, 1)] + LARGE[:2])
def test_wino_u_layouts_agree(gpu, ci, co, l, k, d):
    """u_layout 1 (U transposed, the Kokoro graph's form) runs the same MFMAs in the same order as the reference
    layout: the outputs and statistics are the same bits (small grids through the split-K path too)."""
    lk = gpu
    r, x, w, b = _case(ci + 2 * l + k, l, ci, co, k)
    pad = _pad(k, d)
    u, tr = W.wino_weights(w)
    ut, tr2 = W.wino_weights_t(w)
    n = W.variant(k)[1]
    # the tiled element (x, cb, c, g, k4, j, q) is U[x, g Ci + 16 c + 4 k4 + q, 64 cb + j]
    t = ut.reshape(u.shape[0], co // 64, ci // 16, n, 4, 64, 4)
    x_, cb, c, g, k4, j, q = 1, co // 64 - 1, ci // 16 - 1, n - 1, 2, 37, 3
    assert t[x_, cb, c, g, k4, j, q] == u[x_, g * ci + 16 * c + 4 * k4 + q, 64 * cb + j]
    assert np.array_equal(tr, tr2) and np.array_equal(np.sort(ut.ravel()), np.sort(u.ravel()))
    args = (G(lk, x), None, G(lk, b), G(lk, tr), k)
    y0, s0 = lk.ops.conv1d_wino_lc_f32_gpu(args[0], G(lk, u), *args[2:], padding=pad, dilation=d, stats=True)
    y1, s1 = lk.ops.conv1d_wino_lc_f32_gpu(args[0], G(lk, ut), *args[2:], padding=pad, dilation=d, stats=True,
                                           u_layout=1)
    assert np.array_equal(y0.numpy(), y1.numpy())
    assert np.array_equal(s0.numpy(), s1.numpy())


@pytest.mark.parametrize("ci,co,l,k,d", [(16, 64, 1, 3, 1), (32, 64, 129, 3, 1), (48, 128, 255, 3, 5), (16, 64, 300, 4, 1),
                                         (80, 64, 515, 7, 3), (64, 128, 259, 11, 5), (1104, 1024, 300, 3, 1)])
def test_wino_split_u(gpu, ci, co, l, k, d):
    """u_layout 2 (U in three bf16 parts): the same MFMAs as the other layouts, so the same bits, through every chunk
    count per step (16, 32, 48 channels), one to three tap groups, ragged tiles and the split-K path."""
    lk = gpu
    r, x, w, b = _case(ci + l + 5 * k, l, ci, co, k)
    u, tr = W.wino_weights(w)
    us = lk.ops.wino_split_u_f32_gpu(G(lk, W.wino_weights_t(w)[0]))
    kw = dict(padding=_pad(k, d), dilation=d, stats=True)
    y0, s0 = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), G(lk, u), G(lk, b), G(lk, tr), k, **kw)
    y2, s2 = lk.ops.conv1d_wino_lc_f32_gpu(G(lk, x), us, G(lk, b), G(lk, tr), k, u_layout=2, **kw)
    assert np.array_equal(y0.numpy(), y2.numpy()) and np.array_equal(s0.numpy(), s2.numpy())
    close(y2, _direct(x, w, b, _pad(k, d), d), 2e-4)


def test_wino_split_u_parts(gpu):
    """The parts sum to the value exactly, in fragment order, from denormal-free small to the largest floats."""
    lk = gpu
    r = np.random.default_rng(5)
    ut = (r.standard_normal((2, 2, 2048)) * 10.0 ** r.integers(-25, 25, (2, 2, 2048))).astype(np.float32)
    ut[0, 0, :6] = [np.inf, -np.inf, 3.4e38, -3.4028235e38, 3.39616e38, 0.0]
    us = lk.ops.wino_split_u_f32_gpu(G(lk, ut)).numpy().view(np.uint16).reshape(2, 2, 2, 2, 3, 64, 8)
    p = (us.astype(np.uint32) << 16).view(np.float32)
    with np.errstate(over="ignore", invalid="ignore"):
        back = (p[..., 0, :, :] + p[..., 1, :, :]) + p[..., 2, :, :]  # slab, cb, half, set, lane, k
    back = back.reshape(2, 2, 2, 2, 2, 32, 2, 4).transpose(0, 1, 3, 4, 6, 2, 5, 7)  # set, k8, k4, half, col, k
    assert np.array_equal(back.reshape(ut.shape), ut)


def _mm_exact(v, u, tr, lo, k, a):
    """wino_mm of d = 1 in float64 from its operands: y[t M + j] = sum_xi AT[j, xi] sum_g V[xi, t + g] U[xi, g]."""
    n, co = W.variant(k)[1], u.shape[2]
    v = v.astype(np.float64).reshape(a, -1, v.shape[1])
    t = -(-lo // 4)
    at = tr[a * a:].astype(np.float64).reshape(4, a)
    with np.errstate(all="ignore"):
        m = sum(v[:, g:g + t] @ u[:, g * v.shape[2]:(g + 1) * v.shape[2]].astype(np.float64) for g in range(n))
        y = sum(at[:, x, None, None] * m[x][None] for x in range(a))
    return y.transpose(1, 0, 2).reshape(4 * t, co)[:lo]


@pytest.mark.parametrize("layout", [0, 2])
@pytest.mark.parametrize("ci,l,k", [(32, 300, 3), (48, 150, 11), (1024, 70, 3)])
def test_wino_mm_extreme_operands(gpu, ci, l, k, layout):
    """Operands the three-part split cannot hold (infinities, NaN, values past the largest bf16) give what the f32 sum
    gives, and rows of very different magnitude keep f32's relative error each."""
    lk = gpu
    r, x, w, b = _case(ci + l + k, l, ci, 64, k)
    u, tr = W.wino_weights(w)
    a, n = u.shape[0], W.variant(k)[1]
    us = lk.ops.wino_split_u_f32_gpu(G(lk, W.wino_weights_t(w)[0])) if layout == 2 else G(lk, u)
    kw = dict(dilation=1, groups=n, kernel=k, padding=_pad(k, 1), tile=4)
    rows = W.tiles_rows(l, 1, n, 4, k)
    scale = 10.0 ** r.integers(-15, 15, (1, rows // a, 1))
    base = (r.standard_normal((a, rows // a, ci)) * scale).reshape(rows, ci).astype(np.float32)
    zero = np.zeros(64, np.float32)

    def run(v):
        return lk.ops.wino_mm_lc_f32_gpu(G(lk, v), us, G(lk, zero), G(lk, tr), G(lk, x), u_layout=layout, **kw).numpy()

    ref, got = _mm_exact(base, u, tr, l, k, a), run(base)
    # each output row: n ci products per point and A points summed in f32, bounded by sqrt(n ci A) 2^-24 of the rms of
    # its terms' magnitudes, times 16 for the largest of the row
    at = np.abs(tr[a * a:]).reshape(4, a)
    mag = _mm_exact(np.abs(base), np.abs(u), np.concatenate([tr[:a * a], at.ravel()]), l, k, a)
    assert (np.abs(got - ref).max(1) <= 16 * 2.0 ** -24 * mag.max(1)).all()
    for bad in (np.inf, -np.inf, np.nan, 3.4e38):
        v = base / np.float32(1e15)
        v[rows // a + 3, 5] = bad
        v[2 * (rows // a) + 9, ci - 1] = bad
        ref, got = _mm_exact(v, u, tr, l, k, a), run(v)
        big = np.abs(ref) > 3e38  # overflows in f32
        assert np.array_equal(np.isnan(ref), np.isnan(got))
        ok = np.isfinite(ref) & ~big
        fine = np.where(np.isfinite(v), v, 0)  # what the finite outputs are sums of
        mag = _mm_exact(np.abs(fine), np.abs(u), np.concatenate([tr[:a * a], at.ravel()]), l, k, a)
        assert (np.abs(got[ok] - ref[ok]) <= 2.0 ** -24 * (6 + 2 * np.sqrt(n * ci * a)) * mag[ok]).all()
        inf = np.isinf(ref)
        assert np.array_equal(got[inf], ref[inf].astype(np.float32))


def _mm_operands(lk, r, ci, l, k, tile, d, layout, u=None):
    """A wino_mm call over random operands of 64 output channels: (run(v, u), v, u, tr, exact(v, u)); run launches it
    in the given u_layout, exact is the same in float64."""
    n, a, m = W.variant(k)[1], W.alpha_of(k, tile), 2 if tile == 2 else 4
    tr = W.wino_weights(np.zeros((64, 16, k)), tile)[1]
    rows = W.tiles_rows(l, d, n, tile, k)
    v = r.standard_normal((rows, ci)).astype(np.float32)
    u = r.standard_normal((a, n * ci, 64)).astype(np.float32)
    x, zero = np.zeros((l, ci), np.float32), np.zeros(64, np.float32)
    at = tr[a * a:].astype(np.float64).reshape(m, a)

    def run(v, u):
        dev = G(lk, u if layout == 0 else W.tile_u(u, n))
        dev = lk.ops.wino_split_u_f32_gpu(dev) if layout == 2 else dev
        return lk.ops.wino_mm_lc_f32_gpu(G(lk, v), dev, G(lk, zero), G(lk, tr), G(lk, x), dilation=d, groups=n, kernel=k,
                                         padding=_pad(k, d), tile=tile, u_layout=layout).numpy()

    def exact(v, u, at=at):
        v, u = v.astype(np.float64).reshape(d, a, -1, ci), u.astype(np.float64)
        y = np.zeros((l, 64))
        for rho in range(min(d, l)):
            t = -(-len(range(rho, l, d)) // m)
            p = [sum(v[rho, i, g:g + t] @ u[i, g * ci:(g + 1) * ci] for g in range(n)) for i in range(a)]
            full = np.stack([sum(at[j, i] * p[i] for i in range(a)) for j in range(m)], 1).reshape(m * t, 64)
            y[rho::d] = full[:len(range(rho, l, d))]
        return y

    def bound(v, u):  # of the f32 sum: n ci products per point, A points, random signs
        return 2.0 ** -24 * (6 + 2 * np.sqrt(n * ci * a)) * exact(np.abs(v), np.abs(u), np.abs(at))

    return run, v, u, exact, bound


# every kernel of the launcher: tile 2, one to three chunks of 16 channels per step, two and three tap groups; split-K
# (one residue of a few tiles), dilation
MM_KERNELS = [(32, 200, 3, 2, 1), (16, 90, 3, 4, 2), (32, 300, 3, 4, 1), (48, 300, 3, 4, 3), (32, 200, 7, 4, 3),
              (48, 150, 11, 4, 1), (768, 70, 3, 4, 1)]


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("ci,l,k,tile,d", MM_KERNELS)
def test_wino_mm_largest_products(gpu, ci, l, k, tile, d, layout):
    """A product that f32 holds is not lost where the operands' leading parts, both rounded up, multiply past it."""
    run, v, u, exact, _ = _mm_operands(gpu, np.random.default_rng(1), ci, l, k, tile, d, layout)
    v, u = np.zeros_like(v), np.zeros_like(u)
    top = np.float32(0.9985 * 2.0 ** 64)
    r1 = len(v) // (d * len(u))  # the rows of point 1 (residue 0), whose coefficients AT[:, 1] are all 1
    v[r1 + 3, 5], v[r1 + 10, ci - 1] = top, -top
    u[1, 5, 7], u[1, ci - 1, 40] = top, top
    want = exact(v, u).astype(np.float32)
    assert np.isfinite(want).all() and np.abs(want).max() > 3.39e38
    assert np.array_equal(run(v, u), want)


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("ci,l,k,tile,d", MM_KERNELS)
def test_wino_mm_small_operands(gpu, ci, l, k, tile, d, layout):
    """Operands down to the smallest denormals, all of V or columns of U, enter with all their bits."""
    r = np.random.default_rng(ci + l + k)
    run, v, u, exact, bound = _mm_operands(gpu, r, ci, l, k, tile, d, layout)
    big = np.float32(2.0 ** 60)
    for e in (-112, -127, -145):
        tiny = (v * 2.0 ** e).astype(np.float32)
        assert (np.abs(run(tiny, u * big) - exact(tiny, u * big)) <= bound(tiny, u * big)).all()
    tiny = (u * 2.0 ** -r.integers(100, 148, 64)).astype(np.float32)
    assert (np.abs(run(v * big, tiny) - exact(v * big, tiny)) <= bound(v * big, tiny)).all()


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("ci,l,k,tile,d", MM_KERNELS)
def test_wino_mm_nonfinite_operands(gpu, ci, l, k, tile, d, layout):
    """Infinities, NaN and values past the largest bf16, in V or in U, through every kernel: they reach the outputs that
    the f32 sums take them to, and every finite output of the recomputed tiles is the f32 sum."""
    run, v0, u0, exact, bound = _mm_operands(gpu, np.random.default_rng(ci + l + k), ci, l, k, tile, d, layout)
    r1 = len(v0) // (d * len(u0))
    for bad in (np.inf, -np.inf, np.nan, 3.4e38):
        for where in ("v", "u"):
            v, u = (v0, u0 * np.float32(0.15)) if where == "v" else (v0 * np.float32(0.15), u0)  # no product past 3.4e38
            v, u = v.copy(), u.copy()
            if where == "v":
                v[r1 + 3, 5] = v[(len(u0) - 1) * r1 + 9, ci - 1] = bad
            else:
                u[1, 5, 7] = u[len(u0) - 1, ci - 1, 40] = bad
            with np.errstate(all="ignore"):
                ref, got = exact(v, u), run(v, u)
                lim = bound(np.where(np.isfinite(v), v, 0), np.where(np.isfinite(u), u, 0))
                assert np.array_equal(np.isnan(ref), np.isnan(got))
                inf, ok = np.isinf(ref), np.abs(ref) < 3e38
                assert np.array_equal(got[inf], ref[inf].astype(np.float32))
                assert ok.any() and (np.abs(got[ok] - ref[ok]) <= lim[ok]).all()


@pytest.mark.parametrize("layout", [0, 1, 2])
def test_wino_mm_nan_weights(gpu, layout):
    """Every NaN of U stays one, also with all its significand bits in the low half (the split layout)."""
    run, v, u, _, _ = _mm_operands(gpu, np.random.default_rng(2), 32, 200, 3, 4, 1, layout)
    u.view(np.uint32)[1, 7, 5], u.view(np.uint32)[2, 31, 60] = 0x7f800001, 0xff800001
    y = run(v, u)
    assert np.isnan(y[:, [5, 60]]).all() and np.isfinite(np.delete(y, [5, 60], 1)).all()


@pytest.mark.parametrize("layout", [0, 1, 2])
def test_wino_mm_wide_rows(gpu, layout):
    """Output rows of which 32 take 4 GB (dilation x Co = 2^25): a column block gives the same bits as by itself."""
    import torch

    lk, ci, co, d, l = gpu, 16, 1 << 19, 64, 270  # 4 or 5 rows per residue class
    g = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    tr = lk.Tensor(torch.from_numpy(W.wino_weights(np.zeros((64, 16, 3)))[1]).cuda())
    v, u, b, res = rnd(W.tiles_rows(l, d, 1, 4, 3), ci), rnd(6, ci, co), rnd(co), rnd(l, co)
    x = lk.Tensor(torch.zeros(l, ci, device="cuda"))

    def run(cols):
        n = cols.stop - cols.start
        w = u[:, :, cols]
        if layout:  # winograd.tile_u
            w = w.reshape(6, ci // 16, 4, 4, n // 64, 64).permute(0, 4, 1, 2, 5, 3).reshape(6, n // 64, ci * 64)
        w = lk.Tensor(w.contiguous())
        w = lk.ops.wino_split_u_f32_gpu(w) if layout == 2 else w
        y, st = lk.ops.wino_mm_lc_f32_gpu(lk.Tensor(v), w, lk.Tensor(b[cols]), tr, x, dilation=d, groups=1, kernel=3,
                                          padding=d, tile=4, residual=lk.Tensor(res[:, cols]), out_scale=0.5, stats=True,
                                          u_layout=layout)
        return y.t, st.t

    y, st = run(slice(0, co))
    for c in (0, co // 2, co - 128):
        yc, sc = run(slice(c, c + 128))
        assert torch.equal(y[:, c:c + 128], yc) and torch.equal(st[:, c:c + 128], sc)
