"""The prompt attention (lbd_attention) at the edges of its tiles (GPU): 16-query tiles in
pairs, 16-, 32- and 64-key chunks split over eight waves, caches that end inside a chunk,
addresses that are only 4-byte aligned, and rows that a query must not see.

Bound: scores of D float32 products of |q| |k| <= 25 and a softmax-weighted mean of at
most 1100 values, each sum within (D + 16) 2^-24 of its magnitudes: 2e-5 max|v|, the
bar of test_gpu_model.test_attention."""
import numpy as np
import pytest

from lowbit_amd import kernels as K
from test_gpu_model import attention_ref, ok

pytestmark = pytest.mark.gpu


def attend(q, kc, vc, T, H, KV, D, pos, shift=0):
    """lbd_attention with q, v and out `shift` floats past a 256-byte boundary."""
    L, cap = K.lib(), kc.shape[1]
    pad = lambda a: np.concatenate([np.zeros(shift, np.float32), a.ravel()])  # noqa: E731
    dq, dk, dv = (K.DeviceBuffer.from_array(a) for a in (pad(q), kc, pad(vc)))
    dp, out = K.DeviceBuffer.from_array(np.array([pos], np.int32)), K.DeviceBuffer((T * H * D + shift) * 4)
    ok(L.lbd_attention(dq.ptr + 4 * shift, q.shape[1], dk.ptr, dv.ptr + 4 * shift, T, H, KV, D, dp.ptr, cap,
                       out.ptr + 4 * shift, None))
    return out.to_array((T * H * D + shift,), np.float32)[shift:].reshape(T, H * D)


def draw(rng, T, H, KV, D, cap):
    return (rng.standard_normal((T, (H + 2 * KV) * D)).astype(np.float32),
            rng.standard_normal((KV, cap, D)).astype(np.float32), rng.standard_normal((KV, cap, D)).astype(np.float32))


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("T,H,KV,pos,cap,shift", [
    (1, 2, 1, 0, 1, 0), (16, 3, 1, 0, 16, 1), (17, 4, 2, 15, 40, 2), (32, 2, 2, 0, 32, 0), (33, 7, 1, 31, 64, 3),
    (47, 2, 1, 513, 561, 0), (65, 4, 4, 0, 65, 1), (20, 2, 1, 1080, 1100, 0),
    # few scores over at most 64 positions (104 at D = 128) have a kernel of their own: its last
    # sizes, and the tiles' edges past it
    (64, 12, 4, 0, 64, 1), (64, 13, 1, 0, 64, 0), (5, 2, 1, 59, 64, 0), (40, 3, 1, 64, 104, 1), (33, 32, 4, 16, 49, 1),
    (1, 2, 1, 0, 105, 0), (16, 3, 1, 0, 112, 1), (17, 4, 2, 88, 105, 2), (32, 2, 2, 0, 128, 0), (33, 7, 1, 72, 105, 3),
    (48, 3, 1, 60, 120, 1), (65, 4, 4, 41, 106, 1)])
def test_tile_edges(rng, D, T, H, KV, pos, cap, shift):
    q, kc, vc = draw(rng, T, H, KV, D, cap)
    kc[:, pos + T:], vc[:, pos + T:] = np.nan, np.nan  # cache rows past the keys in use
    got = attend(q, kc, vc, T, H, KV, D, pos, shift)
    ref = attention_ref(q[:, :H * D].reshape(T, H, D), kc, vc, pos, H, KV)
    assert np.abs(got - ref).max() <= 2e-5 * np.nanmax(np.abs(vc))


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("cap", [48, 120])
def test_rows_a_query_does_not_see_may_hold_anything(rng, D, bad, cap):
    """Key 21's value (then key 38's key) is not finite: queries before it are the
    finite attention, queries from it on are not finite (NaN scores and sums)."""
    T, H, KV, pos = 45, 4, 2, 3
    q, kc, vc = draw(rng, T, H, KV, D, cap)
    ref = attention_ref(q[:, :H * D].reshape(T, H, D), kc, vc, pos, H, KV)
    v2 = vc.copy()
    v2[:, 21] = bad
    got = attend(q, kc, v2, T, H, KV, D, pos)
    assert np.abs(got[:21 - pos] - ref[:21 - pos]).max() <= 2e-5 * np.abs(vc).max()
    assert not np.isfinite(got[21 - pos:]).any()
    k2 = kc.copy()
    k2[:, 38] = np.nan
    got = attend(q, k2, vc, T, H, KV, D, pos)
    assert np.abs(got[:38 - pos] - ref[:38 - pos]).max() <= 2e-5 * np.abs(vc).max()
    assert np.isnan(got[38 - pos:]).all()
