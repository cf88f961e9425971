"""Prefill's last-row logits of several sequences where the matrix-core route's
workspace finds no memory (host logic, on a runtime without a device)."""

PREFILL = """
def prefill(vocab, room=1 << 40):
    F.fake_limit(1 << 62)
    cfg = E.LlamaConfig(vocab_size=vocab, hidden_size=4096, intermediate_size=512, n_layers=1, n_heads=32, n_kv_heads=8,
                        max_seq_len=64, rope_theta=10000.0, tie_word_embeddings=False)
    m = E.LlamaModel.new_random(cfg, 1, init_on_device=True)
    caches = [m.new_llama_kv_cache(8) for _ in range(3)]
    F.fake_limit(F.fake_used() + room)
    launches()
    m.prefill(caches, np.zeros((3, 5), np.int64))
    return " ".join(l.split()[0] for l in launches()[-2:])
"""


def test_no_room_for_the_head_workspace(fake_hip):
    out = fake_hip(PREFILL + "print(prefill(128256, 32 << 20), '|', prefill(128256))").split("|")
    assert "k_qgemv" in out[0] and "k_skinny" not in out[0]
    assert "k_skinny" in out[1]
