"""The op-level glue kernels at the edges of their dispatch: a wave or a
workgroup per softmax row and the rows too long for registers, norms with 256
and 1024 threads and ragged widths, 16-byte and single accesses of the data
movers, RoPE's head groups, the two-launch argmax.  References in float64 or
exact; f32 results of f64 sums within one rounding (2^-24 relative) plus, for
softmax, expf's few ulps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("rows,cols", [(3, 1), (5, 63), (1500, 255), (1025, 512), (1024, 777), (1100, 1500), (1024, 2048),
                                       (7, 1001), (9, 2049), (2, 4097), (3, 8192), (2, 9001)])
def test_softmax_rows(hip, rows, cols):
    B = hip.HipBackend
    rng = np.random.default_rng(rows + cols)
    x = rng.normal(0, 4, (rows, cols)).astype(F)
    if cols > 4:
        x[0, 1] = -np.inf
        x[rows - 1, 3] = F(-1e9)
    for scale in (None, 0.125):
        v = (x if scale is None else x * F(scale)).astype(np.float64)
        e = np.exp(v - v.max(1, keepdims=True))
        ref = e / e.sum(1, keepdims=True)
        s = B.from_vec(x)
        out = (B.softmax(s, rows, cols) if scale is None else B.scaled_softmax(s, scale, rows, cols)).to_vec()
        out = out.reshape(rows, cols).astype(np.float64)
        # expf: 2 ulps and the f32 rounding of v - max (2^-24 |v - max|); denormal results absolutely
        tol = (3 * 2.0 ** -23 + 2.0 ** -23 * np.abs(np.where(np.isinf(v), 0, v) - v.max(1, keepdims=True))) * ref + 1e-37
        assert (np.abs(out - ref) <= tol).all()
    y = x.copy()
    y[0, cols // 2] = np.nan
    out = B.softmax(B.from_vec(y), rows, cols).to_vec().reshape(rows, cols)
    assert np.isnan(out[0]).all() and not np.isnan(out[1:]).any()


@pytest.mark.parametrize("rows,d", [(1, 4), (1, 288), (3, 1026), (2, 4096), (300, 4096), (260, 2052), (5, 5120), (2, 16384),
                                    (1, 20000), (257, 768)])
def test_norms(hip, rows, d):
    B = hip.HipBackend
    rng = np.random.default_rng(d)
    x = rng.normal(1, 3, (rows, d)).astype(F)
    g, b = rng.normal(1, 0.2, d).astype(F), rng.normal(0, 0.2, d).astype(F)
    x64 = x.astype(np.float64)
    ref = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + np.float64(F(1e-5))) * g
    out = B.rmsnorm(B.from_vec(x), B.from_vec(g), rows, d, 1e-5).to_vec().reshape(rows, d)
    assert (np.abs(out - ref) <= 2.0 ** -23 * np.abs(ref) + 1e-30).all()
    n = (x64 - x64.mean(1, keepdims=True)) / np.sqrt(x64.var(1, keepdims=True) + np.float64(F(1e-5)))
    ref = n * g + b
    o, mu, rs = B.layernorm(B.from_vec(x), B.from_vec(g), B.from_vec(b), rows, d, 1e-5)
    assert (np.abs(o.to_vec().reshape(rows, d) - ref) <= 2.0 ** -23 * np.abs(ref) + 1e-12).all()
    assert np.allclose(mu.to_vec(), x64.mean(1), rtol=1e-6, atol=1e-9)


@pytest.mark.parametrize("hd", [4, 6, 64])
def test_data_movers(hip, hd):
    B = hip.HipBackend
    rng = np.random.default_rng(hd)
    L, nkv, rep, S = 37, 3, 4, 9
    nq = nkv * rep
    c = rng.normal(size=(L + 5, nkv, hd)).astype(F)
    ref = c[:L].transpose(1, 0, 2).repeat(rep, axis=0)
    assert np.array_equal(B.gather_reshape_repeat_kv(B.from_vec(c), L + 5, L, nkv, nq, hd).to_vec(), ref.ravel())
    k = rng.normal(size=(nkv, S, hd)).astype(F)
    assert np.array_equal(B.repeat_kv(B.from_vec(k), nkv, nq, S, hd).to_vec(), k.repeat(rep, axis=0).ravel())
    x = rng.normal(size=(S, 3, nq, hd)).astype(F)
    for got, want in zip(B.split_qkv_reshape_heads(B.from_vec(x), S, nq, hd), x.transpose(1, 2, 0, 3)):
        assert np.array_equal(got.to_vec(), want.ravel())
    y = rng.normal(size=(2, S, nq, hd)).astype(F)
    r = B.reshape_for_heads(B.from_vec(y), 2, S, nq, hd)
    assert np.array_equal(r.to_vec(), y.transpose(0, 2, 1, 3).ravel())
    assert np.array_equal(B.reshape_from_heads(r, 2, S, nq, hd).to_vec(), y.ravel())
    z = rng.normal(size=(5, 10 * hd)).astype(F)
    for a, w in ((0, hd), (hd, 2 * hd), (3, 5)):
        assert np.array_equal(B.gather_columns(B.from_vec(z), 5, 10 * hd, a, w).to_vec(), z[:, a:a + w].ravel())
    for seq in (1, 5, 8, 300):
        m = rng.normal(size=(3, seq, seq)).astype(F)
        s = B.from_vec(m)
        B.apply_batched_causal_mask_and_scale(s, 3, seq, 0.25, -1e9)
        assert np.array_equal(s.to_vec().reshape(m.shape), np.where(np.tril(np.ones((seq, seq), bool)), m * F(0.25), F(-1e9)))
    for n in (1, 3, 4, 1023, 4096):
        u, v = rng.normal(size=n).astype(F), rng.normal(size=n).astype(F)
        assert np.array_equal(B.add(B.from_vec(u), B.from_vec(v)).to_vec(), u + v)
        assert np.array_equal(B.scale(B.from_vec(u), 0.3).to_vec(), u * F(0.3))


@pytest.mark.parametrize("nh", [1, 6, 8, 9, 32])
def test_rope_head_groups(hip, orc, nh):
    B = hip.HipBackend
    rng = np.random.default_rng(nh)
    x = rng.normal(size=(7, nh, 48)).astype(F)
    fr = (1.0 / 10000.0 ** (np.arange(24) / 24.0)).astype(F)
    got = B.rope_with_freqs_preloaded(B.from_vec(x), 7, nh, 48, 11, B.from_vec(fr)).to_vec().reshape(x.shape)
    ang = (11 + np.arange(7, dtype=np.float64))[:, None, None] * fr.astype(np.float64)
    c, s = np.cos(ang).astype(F), np.sin(ang).astype(F)
    ref = np.stack((x[..., 0::2] * c - x[..., 1::2] * s, x[..., 0::2] * s + x[..., 1::2] * c), -1).reshape(x.shape)
    assert np.abs(got - ref).max() <= 2.0 ** -22 * np.abs(ref).max()  # an f32 ulp of the two libms' cos / sin


@pytest.mark.parametrize("n", [1, 256, 1024, 1025, 50257, 262145, 1000003])
def test_argmax_ranges(hip, n):
    """The last of equal maxima; with NaNs, the argmax after the last of them (generate.rs:167-173)."""
    B = hip.HipBackend
    rng = np.random.default_rng(n)
    x = rng.normal(size=n).astype(F)
    assert B.argmax(B.from_vec(x)) == int(x.argmax())
    for i in {0, n // 3, n // 2, n - 1}:
        x[i] = 9.0
    assert B.argmax(B.from_vec(x)) == n - 1
    if n > 2:
        x[n // 2 + 1] = np.nan
        x[n - 1] = -3.0
        tail = x[n // 2 + 2:]
        want = n // 2 + 2 + (len(tail) - 1 - int(tail[::-1].argmax())) if len(tail) else n // 2 + 1
        assert B.argmax(B.from_vec(x)) == want


@pytest.mark.parametrize("s,nh,hd,pos", [(1, 32, 128, 1000), (37, 9, 64, 0), (5, 1, 2, 3)])
def test_rope_fused_products(hip, s, nh, hd, pos):
    """Which product of a rotated pair is rounded by itself: the sine's, both for
    the even and the odd value (the other way about a sixth of the values differ
    in their last bit).  The products are exact in 64-bit significands and the
    sums nearly always; cos and sin are f64 rounded to f32, by another library."""
    B = hip.HipBackend
    rng = np.random.default_rng(s + nh)
    x = rng.normal(size=(s, nh, hd // 2, 2)).astype(F)
    f = (1.0 / 10000.0 ** (2.0 * np.arange(hd // 2) / hd)).astype(F)
    ang = (pos + np.arange(s, dtype=np.float64))[:, None, None] * f.astype(np.float64)
    c, sn = np.cos(ang).astype(F), np.sin(ang).astype(F)
    L = np.longdouble
    ref = np.stack([(L(1) * x[..., 0] * c - x[..., 1] * sn).astype(F), (L(1) * x[..., 1] * c + x[..., 0] * sn).astype(F)], -1)
    got = B.rope_with_freqs_preloaded(B.from_vec(x.ravel()), s, nh, hd, pos, B.from_vec(f)).to_vec().reshape(x.shape)
    scaled = B.rope_with_freqs_scaled_preloaded(B.from_vec(x.ravel()), s, nh, hd, pos, B.from_vec(f), 0.125).to_vec()
    assert (got != ref).mean() <= 1e-3
    assert np.array_equal(scaled, (got * F(0.125)).ravel())


@pytest.mark.parametrize("rows,cols", [(2, 100), (1100, 513), (3, 8192), (3, 8193), (2, 20000)])
def test_scaled_softmax_rounds_the_scaled_values(hip, rows, cols):
    """x * scale is rounded to f32 before the maximum is taken off: the same bits
    as softmax of the scaled values."""
    B = hip.HipBackend
    x = np.random.default_rng(cols).normal(0, 4, rows * cols).astype(F)
    got = B.scaled_softmax(B.from_vec(x), 0.13, rows, cols).to_vec()
    assert np.array_equal(got, B.softmax(B.from_vec(x * F(0.13)), rows, cols).to_vec())
