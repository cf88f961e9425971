"""Storage blocks are reused after free: values must not depend on what a block
held before, on blocks freed while their work is still queued, or on threads."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


def test_reuse_while_queued(hip):
    """Intermediates freed right after the call that reads them was queued."""
    B = hip.HipBackend
    rng = np.random.default_rng(0)
    n = 1 << 20
    x = rng.normal(size=n).astype(F)
    s = B.from_vec(x)
    ref = x.copy()
    for i in range(40):
        t = B.scale(s, 1.25)
        s = B.add(t, t)  # t is freed by the next round's assignment
        u = B.scale(s, 0.5)
        s = B.scale(u, 0.75)
        ref = ((ref * F(1.25) + ref * F(1.25)) * F(0.5)) * F(0.75)
    assert np.array_equal(s.to_vec(), ref)


def _dirty(B, value):
    """Two free blocks of every size class up to 2 MB ((8 + i) << (e + 5) bytes) that hold `value`."""
    junk = [B.from_vec(np.full((8 + i) << (e + 3), value, F)) for e in range(14) for i in range(8) for _ in range(2)]
    for j in junk:
        j.free()


@pytest.mark.parametrize("m,k,n", [(20, 100, 64), (150, 768, 96), (150, 700, 33)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_results_do_not_depend_on_old_contents(hip, m, k, n, bad):
    """The GEMM planes come from reused blocks and are not cleared: rows past m
    and columns past k are what the block held.  Every block a call can get holds
    NaN or infinities first; integer operands, so the results are exact."""
    print(f"[case] {m} x {k} x {n} {bad}", flush=True)
    B = hip.HipBackend
    rng = np.random.default_rng(m)
    a = rng.integers(-8, 9, (m, k)).astype(F)
    q = rng.integers(-60, 61, (k, n)).astype(np.int8)
    ref = a.astype(np.float64) @ q.astype(np.float64)
    A, W, Wf, sc = B.from_vec(a), B.i8_from_vec(q), B.from_vec(q.astype(F)), B.ones(n * ((k + 31) // 32))

    def bf16():
        B.set_bf16_mode(True)
        try:
            return B.matmul(A, Wf, m, k, n)
        finally:
            B.set_bf16_mode(False)

    for op in (lambda: B.matmul_i8_f32(A, W, 1.0, m, k, n), lambda: B.matmul_i8_f32_block32(A, W, sc, m, k, n), bf16,
               lambda: B.matmul(A, Wf, m, k, n)):
        for _ in range(2):
            _dirty(B, bad)
            assert np.array_equal(op().to_vec().reshape(m, n), ref)


def test_threads(hip):
    B = hip.HipBackend
    bad = []

    def work(i):
        x = np.full(5000 + 37 * i, i + 1, F)
        for r in range(50):
            s = B.from_vec(x)
            y = B.mul_elementwise(B.add(s, s), s).to_vec()
            if not np.array_equal(y, 2 * x * x):
                bad.append((i, r))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
