"""llamd_hip_be_matmul against the oracle's in-order f32 sums, bit for bit, at
the edges of its tiles (64 rows, 1 to 3 columns per wave, strips of 32 in k)
and on rows whose length leaves them 4-byte aligned only."""
import numpy as np
import pytest

import helpers as H
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (64, 4, 32), (65, 5, 33), (63, 3, 31), (70, 1, 64), (129, 9, 95), (1999, 131, 67),
    (2048, 200, 40), (100, 37, 1031)])
def test_matmul_in_order_bit_exact(gpu, m, n, k):
    w = H.sample(m * k, 71)
    x = H.sample(n * k, 72)
    if k > 1:
        x[0] = -0.0
    W, X, out = (gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(x),
                 gpu.DeviceBuffer(m * n * 4))
    L = gpu.lib()
    assert L.llamd_hip_be_matmul(W.ptr, X.ptr, out.ptr, m, n, k) == 0
    assert L.llamd_fwd_sync() == 0
    got = out.download(np.empty((n, m), np.float32))
    for j in range(n):
        want = O.matvec_f32(w, m, k, x[j * k:(j + 1) * k])
        assert np.array_equal(got[j].view(np.uint32), want.view(np.uint32)), j


def test_matmul_keeps_infinities_and_nan_in_their_outputs(gpu):
    """A non-finite value reaches its own row and column only (the staging of
    partial tiles reads neighbouring values, which no output may see)."""
    m, n, k = 66, 5, 37
    w = H.sample(m * k, 73).reshape(m, k)
    x = H.sample(n * k, 74).reshape(n, k)
    w[65, 36], x[4, 36] = np.inf, np.nan
    W, X, out = (gpu.DeviceBuffer.from_array(w), gpu.DeviceBuffer.from_array(x),
                 gpu.DeviceBuffer(m * n * 4))
    L = gpu.lib()
    assert L.llamd_hip_be_matmul(W.ptr, X.ptr, out.ptr, m, n, k) == 0
    assert L.llamd_fwd_sync() == 0
    got = out.download(np.empty((n, m), np.float32))
    assert np.isnan(got[4]).all() and not np.isfinite(got[:4, 65]).any()
    assert np.isfinite(got[:4, :65]).all()
