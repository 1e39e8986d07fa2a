"""The prompt GEMMs (lb_prompt.hip) at the edges of their tiles (GPU): row blocks and
subtiles past the matrix, one and an odd number of K groups, the stage buffers with every
number of groups left over, the largest zero-points, against the float64 oracle within the
bounds that the batch kernels' tests use."""
import ctypes as C

import numpy as np
import pytest

import lowbit_amd as lb
from lowbit_amd import kernels as K
from oracle import cref
from oracle import reference as O
from problems import outlier_int4_problem

pytestmark = pytest.mark.gpu

# M, N, K: ragged M and N, 1, 2, 3, 7 and 8 groups; 33 or more 16 x 16 tiles of Y per CU of
# 256 (each test asserts that its shapes take these kernels, by the rows a workgroup takes)
SHAPES = [(1041, 3100, 128), (645, 5003, 256), (300, 9728, 384), (2090, 2601, 1024)]


def _int4(rng, n, k, asym, zmax=15):
    g = k // 128
    return lb.Int4Weights(rng.integers(0, 256, (n, k // 2), dtype=np.uint8),
                          (rng.standard_normal((n, g)) * 0.05).astype(np.float32),
                          rng.integers(0, zmax + 1, (n, g), dtype=np.uint8) if asym else None, k)


@pytest.mark.parametrize("m,n,k", SHAPES + [(560, 4030, 896)])
@pytest.mark.parametrize("asym,zmax", [(False, 0), (True, 15), (True, 255)])
def test_w4a8(rng, m, n, k, asym, zmax):
    assert K.prompt_tile("w4a8", m, n, k)
    W = _int4(rng, n, k, asym, zmax)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[3] = 0
    y = K.gemm_w4a8(x, lb.to_device(W))
    a = lb.quantize_act_int8(x)
    ref, bound = cref.c_gemm_w4a8(a.xq, a.scale, a.gsum, W.qw, W.scales, W.zeros)
    O.assert_fp_close(y, ref, bound, 1e-5)
    assert np.array_equal(y[3], np.zeros(n, np.float32))


# every tile height with 1, 3, 7, 8 and 9 groups
W8_SHAPES = [(150, 2000, 128, 32), (300, 1500, 384, 32), (160, 4096, 896, 32), (200, 4096, 1152, 32),
             (1041, 3100, 128, 64), (645, 5003, 384, 64), (256, 9728, 896, 64), (700, 4030, 1152, 64),
             (1050, 6000, 128, 128), (1050, 6000, 384, 128), (512, 9728, 896, 128), (2090, 2601, 1024, 128)]


@pytest.mark.parametrize("m,n,k,rows,zmax,wide", [
    s + z for s in W8_SHAPES for z in ((15, False), (64, False), (255, False), (15, True)) if z[0] <= 64 or s[2] == 128])
def test_w4a8_accumulators_are_exact(rng, m, n, k, rows, zmax, wide):
    """With scales of +-1 a row of Y is an integer below 2^24 (9 groups of 128 x 127 x 64 at
    the most; zero-points past 64 with K = 128 only) times the row's scale, rounded once.
    wide: activations and codes at their extremes."""
    assert K.prompt_tile("w4a8", m, n, k) == (rows, 128)
    W = _int4(rng, n, k, True, zmax)
    if zmax == 64:
        W.zeros[::3] = 64
    W.scales[:] = rng.choice([-1.0, 1.0], W.scales.shape)
    x = rng.standard_normal((m, k)).astype(np.float32)
    if wide:
        x = np.sign(x).astype(np.float32)
        W.qw[:] = rng.choice(np.array([0x00, 0xFF], np.uint8), W.qw.shape)
        W.zeros[:] = rng.choice(np.array([0, 15], np.uint8), W.zeros.shape)
    a = lb.quantize_act_int8(x)
    w = W.codes().astype(np.float64) - np.repeat(W.zeros, 128, axis=1)
    acc = a.xq.astype(np.float64) @ (w * np.repeat(W.scales, 128, axis=1)).T  # exact in float64
    assert np.abs(acc).max() < 2 ** 24
    np.testing.assert_array_equal(K.gemm_w4a8(x, lb.to_device(W)), acc.astype(np.float32) * a.scale[:, None])


def test_w4a8_infinities_and_nan(rng):
    """What row-major weights' kernel makes of them, and nothing in other rows."""
    m, n, k = 645, 5003, 384
    assert K.prompt_tile("w4a8", m, n, k)
    W = _int4(rng, n, k, True)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[3, 7], x[20, 300], x[40], x[41, ::2] = np.inf, -np.inf, np.nan, np.nan
    y, ref = K.gemm_w4a8(x, lb.to_device(W)), K.gemm_w4a8(x, W, isa="gfx950-mfma")
    bad = ~np.isfinite(ref)
    assert not bad[[i for i in range(m) if i not in (3, 20, 40, 41)]].any()
    np.testing.assert_array_equal(y[bad], ref[bad])
    a = lb.quantize_act_int8(np.where(np.isfinite(x), x, 0))
    keep = np.isfinite(x).all(1)
    _, bound = cref.c_gemm_w4a8(a.xq, a.scale, a.gsum, W.qw, W.scales, W.zeros)
    assert (np.abs(y[keep] - ref[keep]) <= 2e-5 * bound[keep]).all()


@pytest.mark.parametrize("m,n,k", SHAPES + [(500, 4030, 896), (384, 4099, 2176), (500, 4096, 3200)])
@pytest.mark.parametrize("asym,zmax", [(False, 0), (True, 15), (True, 255)])
def test_w4a16(rng, m, n, k, asym, zmax):
    """Zero-points past 15 rule the t16f8 copy out; elsewhere it gives t16's bits."""
    assert K.prompt_tile("w4a16", m, n, k) == (32, 256)
    W = _int4(rng, n, k, asym, zmax)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[5] *= 1e30
    x[6] *= 1e-30
    D = lb.to_device(W)
    y = K.gemm_w4a16(x, D)
    O.assert_fp_close(y, O.gemm_w4a16_ref(x, W.qw, W.scales, W.zeros), O.fp_bound(x, W.dequantize()), 1e-5)
    assert D.f8_exact() == (zmax <= 15)
    if D.f8_exact():
        qwt8, st = D.tiles_f8()
        L, prm = K.lib(), K._Params(-1, 0, 0, 0, 0, 0, 0)
        dx, dy = K.DeviceBuffer.from_array(x), K.DeviceBuffer(m * n * 4)
        assert L.lbd_gemm_w4a16_t16f8(dx.ptr, m, k, qwt8.ptr, st.ptr, n, dy.ptr, C.byref(prm), None, 0,
                                      None) == K.ISA_GFX950_MFMA
        np.testing.assert_array_equal(dy.to_array((m, n), np.float32), y)


def test_w4a16_infinities_and_nan(rng):
    """A row that holds one is NaN, as in the batch kernel; the others are as without it."""
    m, n, k = 645, 5003, 384
    assert K.prompt_tile("w4a16", m, n, k)
    D = lb.to_device(_int4(rng, n, k, True))
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = K.gemm_w4a16(x, D)
    x[3, 7], x[20, 300], x[41, ::2] = np.inf, -np.inf, np.nan
    y2, keep = K.gemm_w4a16(x, D), np.isfinite(x).all(1)
    assert np.isnan(y2[~keep]).all() and (~keep).sum() == 3
    np.testing.assert_array_equal(y2[keep], y[keep])
    batch = K.gemm_w4a16(x[:32], D)
    assert K.prompt_tile("w4a16", 32, n, k) is None and np.isnan(batch[[3, 20]]).all()


# 1, 2, 3, 7, 8 and 9 groups, the last of one block; 16-row tiles with every number left over
@pytest.mark.parametrize("m,n,k,rows", [s + (32,) for s in [(2090, 6003, 128), (2090, 5003, 256), (900, 9728, 384),
                                                            (700, 4030, 896), (2090, 2601, 1024), (777, 4096, 1056)]] +
                         [(200, 4100, 1152, 16), (190, 4090, 1280, 16), (235, 4089, 1408, 16)])
def test_mxfp4(rng, m, n, k, rows):
    assert K.prompt_tile("mxfp4", m, n, k) == (rows, 256)
    W = lb.MXFP4Weights(rng.integers(0, 256, (n, k // 2), dtype=np.uint8),
                        rng.integers(117, 131, (n, k // 32), dtype=np.uint8), k)
    W.e8m0[0], W.e8m0[1] = 0, 254  # the smallest and the largest scale
    W.e8m0[2, 0] = 255             # NaN
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[4] = 0
    x[5] *= np.float32(2.0 ** 60)
    x[6] *= np.float32(2.0 ** -90)
    x[7, ::31] *= 4096             # large elements beside ordinary ones in every block
    x[8, 1], x[9, 2] = np.inf, np.nan
    y = K.gemm_mxfp4(x, lb.to_device(W))
    assert np.isnan(y[8]).all() and np.isnan(y[9]).all() and np.isnan(y[:, 2]).all()
    keep, cols = np.ones(m, bool), np.ones(n, bool)
    keep[8:10], cols[:3] = False, False
    ref = O.gemm_mxfp4_ref(x[keep], W.qw[cols], W.e8m0[cols])
    bound = O.fp_bound(x[keep], O.dequant_mxfp4(W.qw[cols], W.e8m0[cols]))
    O.assert_fp_close(y[np.ix_(keep, cols)], ref, bound, 1e-5)
    assert np.array_equal(y[4, cols], np.zeros(cols.sum(), np.float32))


def test_columns_that_take_nothing_from_huge_elements(rng):
    """Where a row's few huge elements meet only zero weights, the other elements' products
    must keep the bound, which the huge ones then add nothing to."""
    m, n, k = 512, 4096, 1152
    assert K.prompt_tile("w4a16", m, n, k) and K.prompt_tile("mxfp4", m, n, k)
    x, W = outlier_int4_problem(rng, m, n, k)
    O.assert_fp_close(K.gemm_w4a16(x, lb.to_device(W)), O.gemm_w4a16_ref(x, W.qw, W.scales, W.zeros),
                      O.fp_bound(x, W.dequantize()), 1e-5)
    huge = np.arange(7, k, 97)
    codes = rng.integers(0, 16, (n, k), dtype=np.uint8)
    codes[:, huge] = 0
    W = lb.MXFP4Weights(lb.formats.pack_nibbles(codes, 32), rng.integers(122, 128, (n, k // 32), dtype=np.uint8), k)
    D = lb.to_device(W)
    for amp in (3e4, 3e9, 3e30):
        x = rng.standard_normal((m, k)).astype(np.float32)
        x[::2, huge] *= np.float32(amp)
        O.assert_fp_close(K.gemm_mxfp4(x, D), O.gemm_mxfp4_ref(x, W.qw, W.e8m0), O.fp_bound(x, W.dequantize()), 1e-5)


# one shape of 32-row tiles and one of 16-row ones
MX_SHAPES = [(1300, 4096, 512), (200, 4100, 1280)]


def test_mxfp4_shapes_take_both_tiles():
    assert [K.prompt_tile("mxfp4", *s) for s in MX_SHAPES] == [(32, 256), (16, 256)]


def _mx_limit(x, W, y):
    """Largest error over the bound, with no absolute floor."""
    ref, bound = O.gemm_mxfp4_ref(x, W.qw, W.e8m0), O.fp_bound(x, W.dequantize())
    return (np.abs(y.astype(np.float64) - ref) / (1e-5 * bound + 1e-300)).max()


def _mx_with_workspace(x, D, size):
    """lbd_gemm_mxfp4_t16 with a workspace of that query's size (None: the library's own)."""
    (m, k), n, (qt, et) = x.shape, D.n, D.tiles()
    L, prm = K.lib(), K._Params(-1, 0, 0, 0, 0, 0, 0)
    nb = 0 if size is None else getattr(L, size)(*((m, k) if size.endswith("bytes") else (1, m, n, k)))
    dx, dy, ws = K.DeviceBuffer.from_array(x), K.DeviceBuffer(m * n * 4), K.DeviceBuffer(nb) if nb else None
    assert L.lbd_gemm_mxfp4_t16(dx.ptr, m, k, qt.ptr, et.ptr, n, dy.ptr, C.byref(prm), ws.ptr if ws else None, nb,
                                None) == K.ISA_GFX950_MFMA
    return dy.to_array((m, n), np.float32)


@pytest.mark.parametrize("m,n,k", MX_SHAPES)
@pytest.mark.parametrize("small", [1, 2, 3, 31])
@pytest.mark.parametrize("amp", [1e6, 1e9, 1e12, 3e38])
def test_mxfp4_small_elements_beside_a_large_one(rng, m, n, k, small, amp):
    """A large element that meets zero weights, `small` ordinary or tiny ones and zeros in
    each block of 32: the products of the small ones must keep the bound."""
    x = np.zeros((m, k // 32, 32), np.float32)
    x[:, :, 0] = amp
    x[:, :, 1:1 + small] = rng.standard_normal((m, k // 32, small))
    x[::3, :, 1:1 + small] *= 1e-10
    x = x.reshape(m, k)
    codes = rng.integers(0, 16, (n, k), dtype=np.uint8)
    codes[:, ::32] = 0
    W = lb.MXFP4Weights(lb.formats.pack_nibbles(codes, 32), rng.integers(122, 128, (n, k // 32), dtype=np.uint8), k)
    assert _mx_limit(x, W, K.gemm_mxfp4(x, lb.to_device(W))) <= 1.0


@pytest.mark.parametrize("m,n,k", MX_SHAPES)
@pytest.mark.parametrize("mag", [1e-36, 1e-33, 1e-30, 1e-10, 1e10, 1e30])
def test_mxfp4_activation_magnitudes(rng, m, n, k, mag):
    """test_gpu_random_shapes.test_activation_magnitudes at prompt sizes. At 1e-36 the
    smallest of the three bf16 terms are subnormal and flushed, and the largest error of 10^6
    outputs comes to the bound (1.03 of it at 1300 x 4096): there the result is held to the
    batch kernel's largest error, whose terms marked blocks take, with a tenth for sums in
    another order."""
    W = lb.quantize_mxfp4(rng.standard_normal((n, k)).astype(np.float32))
    x = (rng.standard_normal((m, k)) * mag).astype(np.float32)
    D = lb.to_device(W)
    limit = 1.0 if mag > 1e-36 else 1.1 * _mx_limit(x, W, _mx_with_workspace(x, D, "lbd_bf16x3_workspace_bytes"))
    assert _mx_limit(x, W, K.gemm_mxfp4(x, D)) <= limit


@pytest.mark.parametrize("m,n,k", MX_SHAPES + [(528, 4100, 8320), (200, 4100, 8320)])  # 65 groups too
@pytest.mark.parametrize("mag", [1e-20, 1.0, 1e30])
def test_mxfp4_keeps_every_bit_of_an_activation(rng, m, n, k, mag):
    """Weight rows with a single 1: y[i, j] is one of row i's activations itself, normal or
    log-uniform over 2^40, whatever its neighbours are. (All above 2^-110: below it the last
    of an activation's three bf16 terms would be a subnormal, which the matrix cores flush,
    2^-16 of the element at the most, in the batch kernel as here.)"""
    assert K.prompt_tile("mxfp4", m, n, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[m // 2:] *= np.exp2(rng.uniform(-20, 20, x[m // 2:].shape)).astype(np.float32)
    x *= np.float32(mag)
    codes = np.zeros((n, k), np.uint8)
    col = np.arange(n) % k
    col[::2] = k - 1 - col[::2]
    codes[np.arange(n), col] = 2  # E2M1 1.0
    W = lb.MXFP4Weights(lb.formats.pack_nibbles(codes, 32), np.full((n, k // 32), 127, np.uint8), k)
    np.testing.assert_array_equal(K.gemm_mxfp4(x, lb.to_device(W)), x[:, col])


@pytest.mark.parametrize("m,n,k", MX_SHAPES)
def test_mxfp4_rows_do_not_depend_on_each_other(rng, m, n, k):
    """Outliers, tiny values, infinities and NaN in some rows leave the others' bits alone
    (weight rows with few nonzeros, so that the lowest bits of an activation show)."""
    codes = rng.integers(0, 16, (n, k), dtype=np.uint8) * (rng.random((n, k)) < 2 / k).astype(np.uint8)
    W = lb.MXFP4Weights(lb.formats.pack_nibbles(codes, 32), rng.integers(120, 130, (n, k // 32), dtype=np.uint8), k)
    D = lb.to_device(W)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[m // 2:, ::5] *= np.exp2(rng.uniform(-30, 10, (m - m // 2, (k + 4) // 5))).astype(np.float32)
    y = K.gemm_mxfp4(x, D)
    x2, hit = x.copy(), np.arange(m) % 7 == 3
    x2[hit, ::9] *= 1e9
    x2[3], x2[10, 4], x2[17, 5] = 1e-38, np.inf, np.nan
    y2 = K.gemm_mxfp4(x2, D)
    np.testing.assert_array_equal(y2[~hit], y[~hit])
    assert not np.array_equal(y2[hit], y[hit])


@pytest.mark.parametrize("shift", [0, 1])
def test_mxfp4_y_on_x(rng, shift):
    """Y may lie on X (N = K), or begin in X's last row: marked blocks are read from X while
    Y is stored, so such a call takes the batch kernel, which is done with X by then."""
    m, n = 1040, 2048
    assert K.prompt_tile("mxfp4", m, n, n)
    W = lb.quantize_mxfp4(rng.standard_normal((n, n)).astype(np.float32))
    x = rng.standard_normal((m, n)).astype(np.float32)
    x[:, ::9] *= 1e9
    qt, et = lb.to_device(W).tiles()
    L, prm = K.lib(), K._Params(-1, 0, 0, 0, 0, 0, 0)
    def call(px, py, nb):
        ws = K.DeviceBuffer(nb)
        assert L.lbd_gemm_mxfp4_t16(px, m, n, qt.ptr, et.ptr, n, py, C.byref(prm), ws.ptr, nb,
                                    None) == K.ISA_GFX950_MFMA
    dx, dy = K.DeviceBuffer.from_array(x), K.DeviceBuffer(m * n * 4)
    call(dx.ptr, dy.ptr, L.lbd_bf16x3_workspace_bytes(m, n))
    both = K.DeviceBuffer.from_array(np.concatenate([x, np.zeros_like(x)]))
    off = shift * (m - 1) * n
    call(both.ptr, both.ptr + 4 * off, L.lbd_bf16x3_workspace_bytes_split(1, m, n, n))
    got = both.to_array((2 * m * n,), np.float32)[off:off + m * n].reshape(m, n)
    np.testing.assert_array_equal(got, dy.to_array((m, n), np.float32))


def test_mxfp4_workspace_without_room_for_the_digits_takes_the_batch_kernel(rng):
    """A workspace of lbd_bf16x3_workspace_bytes is accepted and meets the bound; one of
    lbd_bf16x3_workspace_bytes_split gives the bits of the library's own."""
    m, n, k = MX_SHAPES[0]
    W = lb.quantize_mxfp4(rng.standard_normal((n, k)).astype(np.float32))
    x = rng.standard_normal((m, k)).astype(np.float32)
    D = lb.to_device(W)
    ys = [_mx_with_workspace(x, D, q) for q in (None, "lbd_bf16x3_workspace_bytes_split", "lbd_bf16x3_workspace_bytes")]
    assert max(_mx_limit(x, W, y) for y in ys) <= 1.0
    np.testing.assert_array_equal(ys[0], ys[1])
    assert not np.array_equal(ys[0], ys[2])
