"""The digit GEMM's tiles and k splits (matmul_i8_f32 above 16 rows, the int8
model's prefill): small integer activations have exact digit planes, so every
tile and split must give the exact integer sums; and a model whose prefill
GEMMs split k against its token-by-token decode."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("m,k,n", [
    (17, 64, 5), (33, 100, 131), (32, 2048, 128), (37, 4096, 260), (64, 768, 768), (65, 3072, 770),
    (130, 4096, 1030), (200, 768, 2304), (129, 8192, 4096), (300, 1024, 4097), (512, 2048, 2050),
    (129, 256, 28416), (600, 128, 28000), (255, 192, 21889), (1100, 64, 13000),
    (384, 1100, 22018), (600, 1024, 14339), (1500, 1024, 6145), (511, 2048, 22013)])
def test_exact_sums(hip, m, k, n):
    print(f"[case] {m} x {k} x {n}", flush=True)
    B = hip.HipBackend
    rng = np.random.default_rng(m + k + n)
    a = rng.integers(-8, 9, (m, k)).astype(F)
    q = rng.integers(-127, 128, (k, n)).astype(np.int8)
    bias = rng.integers(-100, 100, n).astype(F)
    ref = a.astype(np.float64) @ q.astype(np.float64)  # below 2^24: exact in f32
    A, W = B.from_vec(a), B.i8_from_vec(q)
    assert np.array_equal(B.matmul_i8_f32(A, W, 1.0, m, k, n).to_vec().reshape(m, n), ref)
    assert np.array_equal(B.matmul_i8_f32_bias(A, W, 1.0, B.from_vec(bias), m, k, n).to_vec().reshape(m, n), ref + bias)


def test_nonfinite_row_only(hip):
    """A row holding an infinity is NaN as a whole, its neighbours are untouched (k splits included)."""
    B = hip.HipBackend
    m, k, n = 40, 4096, 256
    rng = np.random.default_rng(3)
    a = rng.integers(-8, 9, (m, k)).astype(F)
    q = rng.integers(-127, 128, (k, n)).astype(np.int8)
    ref = a.astype(np.float64) @ q.astype(np.float64)
    a[7, 100] = np.inf
    c = B.matmul_i8_f32(B.from_vec(a), B.i8_from_vec(q), 1.0, m, k, n).to_vec().reshape(m, n)
    assert np.isnan(c[7]).all()
    keep = np.arange(m) != 7
    assert np.array_equal(c[keep], ref[keep])


@pytest.mark.parametrize("seq", [18, 70, 130])
def test_prefill_with_split_k_matches_decode(hip, seq):
    """hidden 2048, ffn 4100: the residual and SwiGLU epilogues after k splits
    (ffn not a multiple of 8), logits within 1e-3 of the decode path's."""
    print(f"[case] seq={seq}", flush=True)
    cfg = hip.LlamaConfig(vocab_size=96, hidden_size=2048, intermediate_size=4100, n_layers=1, n_heads=16,
                          n_kv_heads=4, max_seq_len=256, rope_theta=10000.0, tie_word_embeddings=False)
    m = hip.LlamaModel.new_random(cfg, 3, init_on_device=True)
    toks = np.random.default_rng(seq).integers(0, 96, seq)
    cp, cd = m.new_llama_kv_cache(seq), m.new_llama_kv_cache(seq)
    last = m.prefill([cp], toks[None, :])[0]
    for p, t in enumerate(toks):
        ref, _ = m.forward_with_llama_cache(int(t), p, cd)
    assert np.abs(last - ref).max() <= 1e-3 * np.abs(ref).max()
    m.free()


@pytest.mark.parametrize("mode", ["per_tensor", "block32", "bf16"])
@pytest.mark.parametrize("seq,ffn", [(600, 7172), (384, 11004)])
def test_prefill_in_two_launches_matches_shorter(hip, mode, seq, ffn):
    """SwiGLU columns cut into two launches (full rounds of the chip, the rest):
    one prompt, against the same prompt in pieces of 100 rows, which need no
    cut.  Tolerances as the tests against the decode path."""
    print(f"[case] {mode} seq={seq} ffn={ffn}", flush=True)
    import esolearn_amd.llama as EL
    q = {"per_tensor": EL.QUANT_PER_TENSOR, "block32": EL.QUANT_BLOCK32, "bf16": EL.QUANT_BF16}[mode]
    cfg = hip.LlamaConfig(vocab_size=96, hidden_size=2048, intermediate_size=ffn, n_layers=2, n_heads=16,
                          n_kv_heads=4, max_seq_len=640, rope_theta=10000.0, tie_word_embeddings=False)
    m = hip.LlamaModel.new_random(cfg, 3, quant_mode=q, init_on_device=True)
    toks = np.random.default_rng(seq).integers(0, 96, seq)
    ca, cb = m.new_llama_kv_cache(seq + 1), m.new_llama_kv_cache(seq + 1)
    m.prefill([ca], toks[None, :])
    for at in range(0, seq, 100):
        m.prefill([cb], toks[None, at:at + 100])
    a, _ = m.forward_with_llama_cache(5, seq, ca)  # reads every row of both layers' caches
    b, _ = m.forward_with_llama_cache(5, seq, cb)
    assert np.abs(a - b).max() <= (1e-2 if mode == "bf16" else 1e-3) * np.abs(b).max()
    m.free()


@pytest.mark.parametrize("m,k,n", [
    (17, 64, 5), (37, 100, 131), (32, 4096, 260), (64, 768, 768), (130, 4096, 1030), (200, 3072, 770),
    (129, 1280, 5120), (300, 1024, 4097), (512, 8192, 1024), (600, 2048, 14339)])
def test_bf16_exact_sums(hip, m, k, n):
    """The bf16 GEMM's tiles and splits: integers exact in bf16, sums exact in f32."""
    print(f"[case] bf16 {m} x {k} x {n}", flush=True)
    B = hip.HipBackend
    rng = np.random.default_rng(m + k + n)
    a = rng.integers(-8, 9, (m, k)).astype(F)
    w = rng.integers(-64, 65, (k, n)).astype(F)
    ref = a.astype(np.float64) @ w.astype(np.float64)
    B.set_bf16_mode(True)
    try:
        c = B.matmul(B.from_vec(a), B.from_vec(w), m, k, n).to_vec().reshape(m, n)
    finally:
        B.set_bf16_mode(False)
    assert np.array_equal(c, ref)


@pytest.mark.parametrize("seq", [18, 70, 130])
def test_bf16_prefill_small_tiles_match_decode(hip, seq):
    """The residual splits and the SwiGLU planes of the smaller bf16 tiles, against
    the decode path (both round activations to bf16; one rounding apart at most
    per value: 1e-2 as the bf16 model's other prefill tests)."""
    print(f"[case] bf16 seq={seq}", flush=True)
    import esolearn_amd.llama as EL
    cfg = hip.LlamaConfig(vocab_size=96, hidden_size=2048, intermediate_size=4104, n_layers=1, n_heads=16,
                          n_kv_heads=4, max_seq_len=256, rope_theta=10000.0, tie_word_embeddings=False)
    m = hip.LlamaModel.new_random(cfg, 3, quant_mode=EL.QUANT_BF16, init_on_device=True)
    toks = np.random.default_rng(seq).integers(0, 96, seq)
    cp, cd = m.new_llama_kv_cache(seq), m.new_llama_kv_cache(seq)
    last = m.prefill([cp], toks[None, :])[0]
    for p, t in enumerate(toks):
        ref, _ = m.forward_with_llama_cache(int(t), p, cd)
    assert np.abs(last - ref).max() <= 1e-2 * np.abs(ref).max()
    m.free()


@pytest.mark.parametrize("m,k,n", [
    (17, 64, 5), (33, 100, 131), (40, 4096, 260), (64, 768, 768), (130, 3000, 1030), (129, 4096, 4096),
    (300, 1024, 4097), (512, 11008, 516), (600, 1024, 14339)])
def test_block32_exact_sums(hip, m, k, n):
    """Block-32 scales that are powers of two: every product and sum is exact in f32."""
    print(f"[case] block32 {m} x {k} x {n}", flush=True)
    B = hip.HipBackend
    rng = np.random.default_rng(m + k + n)
    nb = (k + 31) // 32
    a = rng.integers(-3, 4, (m, k)).astype(F)
    q = rng.integers(-40, 41, (k, n)).astype(np.int8)
    s = (2.0 ** rng.integers(-2, 2, (n, nb))).astype(F)
    w = q * s.repeat(32, axis=1)[:, :k].T.astype(np.float64)
    c = B.matmul_i8_f32_block32(B.from_vec(a), B.i8_from_vec(q), B.from_vec(s), m, k, n).to_vec().reshape(m, n)
    assert np.array_equal(c, a.astype(np.float64) @ w)


@pytest.mark.parametrize("seq", [18, 130])
def test_block32_prefill_matches_decode(hip, seq):
    print(f"[case] block32 seq={seq}", flush=True)
    import esolearn_amd.llama as EL
    cfg = hip.LlamaConfig(vocab_size=96, hidden_size=2048, intermediate_size=4100, n_layers=1, n_heads=16,
                          n_kv_heads=4, max_seq_len=256, rope_theta=10000.0, tie_word_embeddings=False)
    m = hip.LlamaModel.new_random(cfg, 3, quant_mode=EL.QUANT_BLOCK32, init_on_device=True)
    toks = np.random.default_rng(seq).integers(0, 96, seq)
    cp, cd = m.new_llama_kv_cache(seq), m.new_llama_kv_cache(seq)
    last = m.prefill([cp], toks[None, :])[0]
    for p, t in enumerate(toks):
        ref, _ = m.forward_with_llama_cache(int(t), p, cd)
    assert np.abs(last - ref).max() <= 1e-3 * np.abs(ref).max()
    m.free()
