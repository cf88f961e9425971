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


@pytest.mark.parametrize("m,k,n", [(20, 100, 64), (150, 768, 96)])
def test_results_do_not_depend_on_old_contents(hip, m, k, n):
    """The GEMM planes come from reused blocks: fill such blocks with NaN and
    infinities first (rows past m and columns past k are theirs)."""
    B = hip.HipBackend
    rng = np.random.default_rng(m)
    a = rng.normal(size=(m, k)).astype(F)
    q = rng.integers(-127, 128, (k, n)).astype(np.int8)
    A, W = B.from_vec(a), B.i8_from_vec(q)
    sc = B.from_vec(np.ones(n * ((k + 31) // 32), F))
    ref = [B.matmul_i8_f32(A, W, 0.1, m, k, n).to_vec(), B.matmul_i8_f32_block32(A, W, sc, m, k, n).to_vec()]
    for bad in (np.nan, np.inf):
        junk = [B.from_vec(np.full(1 << e, bad, F)) for e in range(8, 20) for _ in range(2)]
        junk += [B.from_vec(np.full(3 << e, bad, F)) for e in range(8, 20)]
        for j in junk:
            j.free()
        assert np.array_equal(B.matmul_i8_f32(A, W, 0.1, m, k, n).to_vec(), ref[0])
        assert np.array_equal(B.matmul_i8_f32_block32(A, W, sc, m, k, n).to_vec(), ref[1])


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
