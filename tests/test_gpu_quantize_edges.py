"""The weight quantizers' load paths (GPU), byte for byte against the host packers: 16-byte
loads of aligned rows (K % 4 == 0) and at any float's address elsewhere, rows that end inside
such a load, inside a wave's 512 elements and inside either half of a group, and byte stores
to an unaligned packed array."""
import numpy as np
import pytest

import lowbit_amd as lb
from lowbit_amd import kernels as K

pytestmark = pytest.mark.gpu

KS = [1, 4, 17, 36, 68, 127, 132, 508, 512, 516, 1000, 1001, 1536 + 96]


@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("shift", [0, 1])
def test_ragged_and_unaligned(rng, k, shift):
    """shift: w starts 4 bytes and qw 1 byte past an aligned address."""
    n = 5
    w = rng.standard_normal((n, k)).astype(np.float32)
    w[2] = 0
    L = K.lib()
    buf = K.DeviceBuffer.from_array(np.concatenate([np.zeros(shift, np.float32), w.ravel()]))
    wp = buf.ptr + 4 * shift
    for group, fn in ((128, L.lbd_quantize_int4), (32, L.lbd_quantize_int4_g32)):
        for kw in (dict(), dict(asym=True), dict(scale="signed-max")):
            ref = lb.quantize_int4(w, group=group, **kw)
            qw, s = K.DeviceBuffer(ref.qw.size + 16), K.DeviceBuffer(ref.scales.nbytes)
            z = K.DeviceBuffer(ref.scales.size)
            asym, sm = int("asym" in kw), int("scale" in kw)
            assert fn(wp, n, k, asym, sm, qw.ptr + shift, s.ptr, z.ptr if asym else None, None) == 0
            got = qw.to_array((ref.qw.size + 16,), np.uint8)[shift:shift + ref.qw.size].reshape(ref.qw.shape)
            np.testing.assert_array_equal(got, ref.qw)
            np.testing.assert_array_equal(s.to_array(ref.scales.shape, np.float32), ref.scales)
            if asym:
                np.testing.assert_array_equal(z.to_array(ref.zeros.shape, np.uint8), ref.zeros)
    ref = lb.quantize_mxfp4(w)
    qw, e = K.DeviceBuffer(ref.qw.size + 16), K.DeviceBuffer(ref.e8m0.size)
    assert L.lbd_quantize_mxfp4(wp, n, k, qw.ptr + shift, e.ptr, None) == 0
    got = qw.to_array((ref.qw.size + 16,), np.uint8)[shift:shift + ref.qw.size].reshape(ref.qw.shape)
    np.testing.assert_array_equal(got, ref.qw)
    np.testing.assert_array_equal(e.to_array(ref.e8m0.shape, np.uint8), ref.e8m0)
