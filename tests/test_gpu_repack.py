"""Weight repacks on first use (int8 [k][n] to GEMV rows, bf16 [k][n] to rows):
with a one-hot activation row per k the matmul returns the weight itself."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("k,n", [(1, 16), (16, 16), (130, 128), (127, 144), (300, 400), (129, 20), (64, 17), (1030, 272)])
def test_int8_rows(hip, k, n):
    B = hip.HipBackend
    q = np.random.default_rng(k + n).integers(-128, 128, (k, n)).astype(np.int8)
    s = B.i8_from_vec(q)
    for p in {0, 1 % k, k // 2, max(0, k - 17), k - 1}:
        x = np.zeros(k, F)
        x[p] = 1.0
        assert np.array_equal(B.matmul_i8_f32(B.from_vec(x), s, 1.0, 1, k, n).to_vec(), q[p].astype(F)), p
    m = min(k, 40)
    eye = np.eye(m, k, k - m).astype(F)  # the last m rows
    assert np.array_equal(B.matmul_i8_f32(B.from_vec(eye), s, 1.0, m, k, n).to_vec().reshape(m, n), q[k - m:].astype(F))


@pytest.mark.parametrize("k,n", [(1, 4), (64, 64), (65, 68), (130, 260), (300, 33), (1000, 128)])
def test_bf16_rows(hip, k, n):
    B = hip.HipBackend
    w = np.random.default_rng(k).integers(-128, 129, (k, n)).astype(F)  # exact in bf16
    bits = (w.view(np.uint32) >> 16).astype(np.uint16)
    B.set_bf16_mode(True)
    try:
        s = B.from_vec_with_bf16(w, bits)
        m = min(k, 70)
        for r0 in {0, k - m}:
            eye = np.eye(m, k, r0).astype(F)
            assert np.array_equal(B.matmul(B.from_vec(eye), s, m, k, n).to_vec().reshape(m, n), w[r0:r0 + m])
    finally:
        B.set_bf16_mode(False)
