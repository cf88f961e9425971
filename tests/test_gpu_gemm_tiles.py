"""The GEMMs' tiles and k splits (matmul_i8_f32 and bf16 matmul above 16 rows,
prefill): with integer operands every tile and split must give the exact sums;
prefill's residual and SwiGLU epilogues against the token-by-token decode.
test_gemm_tiles_covered.py holds that the shapes here reach every tile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("m,k,n", [
    (17, 64, 5), (33, 100, 131), (32, 2048, 128), (37, 4096, 260), (64, 768, 768), (65, 3072, 770),
    (130, 4096, 1030), (200, 768, 2304), (129, 8192, 4096), (300, 1024, 4097), (512, 2048, 2050),
    (129, 256, 28416), (600, 128, 28000), (255, 192, 21889), (1100, 64, 13000),
    (384, 1100, 22018), (600, 1024, 14339), (1500, 1024, 6145), (511, 2048, 22013),
    (174, 40, 11339), (77, 6434, 5879), (1416, 51, 681), (1183, 1997, 5), (293, 3552, 6531)])
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
    (129, 1280, 5120), (300, 1024, 4097), (512, 8192, 1024), (600, 2048, 14339),
    (174, 40, 11339), (67, 4864, 2815), (22, 47, 16838), (17, 2240, 2559), (178, 5451, 11150)])
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
    (300, 1024, 4097), (512, 11008, 516), (600, 1024, 14339),
    (174, 40, 11339), (1416, 51, 681), (1183, 1997, 5), (695, 2946, 6226)])
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


PREFILL_SHAPES = [  # weights, hidden, ffn, prompt
    ("per_tensor", 128, 370, 21), ("per_tensor", 1024, 128, 19), ("per_tensor", 2560, 1152, 36), ("per_tensor", 128, 1152, 583),
    ("per_tensor", 128, 4800, 210), ("per_tensor", 128, 4800, 456), ("per_tensor", 2560, 104, 842), ("per_tensor", 640, 8704, 886),
    ("per_tensor", 2176, 8910, 117), ("per_tensor", 3072, 126, 333), ("per_tensor", 2944, 260, 394),
    ("per_tensor", 1216, 62, 804), ("per_tensor", 4096, 2730, 2040),
    ("block32", 128, 370, 26), ("block32", 128, 862, 20), ("block32", 2560, 104, 45), ("block32", 2432, 110, 125),
    ("block32", 128, 4800, 303), ("block32", 128, 3546, 139), ("block32", 384, 2324, 420), ("block32", 384, 2324, 1279),
    ("block32", 2432, 110, 510), ("block32", 2432, 110, 1140), ("block32", 4224, 2046, 34), ("block32", 4096, 512, 2040),
    ("bf16", 128, 448, 19), ("bf16", 128, 1152, 26), ("bf16", 2560, 104, 17), ("bf16", 2432, 110, 39), ("bf16", 128, 862, 615),
    ("bf16", 128, 4800, 88), ("bf16", 256, 1758, 707), ("bf16", 2432, 110, 391), ("bf16", 2560, 104, 413), ("bf16", 2816, 426, 169),
    ("bf16", 2688, 142, 934), ("bf16", 128, 4800, 649), ("bf16", 4096, 512, 2040),
]


def prefill_model(E, mode, h, ffn, seq):
    import esolearn_amd.llama as EL
    q = {"per_tensor": EL.QUANT_PER_TENSOR, "block32": EL.QUANT_BLOCK32, "bf16": EL.QUANT_BF16}[mode]
    nh = h // (64 if h % 128 else 128)
    cfg = E.LlamaConfig(vocab_size=96, hidden_size=h, intermediate_size=ffn, n_layers=2, n_heads=nh,
                        n_kv_heads=nh if nh % 2 else nh // 2, max_seq_len=2048, rope_theta=10000.0,
                        tie_word_embeddings=False)
    return E.LlamaModel.new_random(cfg, 3, quant_mode=q, init_on_device=True)


@pytest.mark.parametrize("mode,h,ffn,seq", PREFILL_SHAPES)
def test_prefill_rows_match_decode(hip, mode, h, ffn, seq):
    """Every row of the second layer's K and V (the first layer's residual and
    SwiGLU epilogues, all columns mixed by K's and V's products) against the
    decode path.  Per row, relative in 2-norm: 1e-3 as the other prefill tests;
    bf16: in each of the four products of a layer a value may round to the other
    neighbour, 2^-8 of it, in quadrature 8e-3.  One wrong column would be 1 /
    sqrt(columns), 1e-2 or more."""
    print(f"[case] {mode} h={h} ffn={ffn} seq={seq}", flush=True)
    m = prefill_model(hip, mode, h, ffn, seq)
    toks = np.random.default_rng(seq).integers(0, 96, seq)
    cp, cd = m.new_llama_kv_cache(seq), m.new_llama_kv_cache(seq)
    m.prefill([cp], toks[None, :])
    for p, t in enumerate(toks):
        m.forward_with_llama_cache(int(t), p, cd)
    for a, b in zip(cp.layer(1), cd.layer(1)):
        a, b = a.reshape(seq, -1).astype(np.float64), b.reshape(seq, -1).astype(np.float64)
        err = np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)
        print(f"[err] {err.max():.2e}", flush=True)
        assert err.max() <= (8e-3 if mode == "bf16" else 1e-3)
    m.free()


@pytest.mark.parametrize("kind", ["bf16", "block32", "per_tensor"])
def test_planes_above_2_gib(hip, kind):
    """More activation bytes than a buffer resource reaches: the register-staged
    kernel (per_tensor: only k above the digit kernel's)."""
    print(f"[case] {kind}", flush=True)
    B = hip.HipBackend
    rows, reps, n = 513, 256, 70
    k = 16448 if kind == "per_tensor" else 8224
    m = rows * reps if kind != "per_tensor" else rows * reps // 2
    rng = np.random.default_rng(k)
    a = rng.integers(-3, 4, (rows, k)).astype(F)
    q = rng.integers(-40, 41, (k, n)).astype(np.int8)
    A = B.repeat_kv(B.from_vec(a), 1, m // rows, rows, k)  # the rows again and again
    if kind == "bf16":
        B.set_bf16_mode(True)
        try:
            c = B.matmul(A, B.from_vec(q.astype(F)), m, k, n)
        finally:
            B.set_bf16_mode(False)
    elif kind == "block32":
        c = B.matmul_i8_f32_block32(A, B.i8_from_vec(q), B.ones(n * ((k + 31) // 32)), m, k, n)
    else:
        c = B.matmul_i8_f32(A, B.i8_from_vec(q), 1.0, m, k, n)
    ref = (a.astype(np.float64) @ q.astype(np.float64)).astype(F)  # below 2^24: exact
    assert np.array_equal(c.to_vec().reshape(-1, rows, n), np.broadcast_to(ref, (m // rows, rows, n)))
