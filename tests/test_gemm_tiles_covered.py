"""The shapes of test_gpu_gemm_tiles.py launch every instantiation of the GEMMs
that the host's choice of tile and k splits can reach (run on a runtime without
a device, which records the launches): a change of the cost model that leaves a
tile without a test fails here."""
import json

RUN = """
import json, os, re
os.environ["SCRY_HIP_NO_GRAPH"] = "1"
sys.path.insert(0, "tests")
import test_gpu_gemm_tiles as T
F.fake_copies(0)
KERNEL = re.compile(r"k_gemm(?:_digits|_ring)?I.*")
seen = set()
def record():
    names = [l.split()[0] for l in launches()]
    for i, n in enumerate(names):
        k = KERNEL.search(n)
        if k:
            seen.add((k.group(), i + 1 < len(names) and "_finish" in names[i + 1]))
def shapes(test):
    return next(m.args[1] for m in test.pytestmark if m.args[0] == "m,k,n")
def matmul(kind, m, k, n):
    A = B.zeros(m * k)
    if kind == "bf16":
        W = B.zeros(k * n)
        B.set_bf16_mode(True)
        B.matmul(A, W, m, k, n)
        B.set_bf16_mode(False)
    else:
        W = B.i8_from_vec(np.empty(k * n, np.int8))
        if kind == "block32":
            B.matmul_i8_f32_block32(A, W, B.zeros(n * ((k + 31) // 32)), m, k, n)
        else:
            B.matmul_i8_f32(A, W, 1.0, m, k, n)
    record()
launches()
for test, kind in ((T.test_exact_sums, "int8"), (T.test_bf16_exact_sums, "bf16"), (T.test_block32_exact_sums, "block32")):
    for s in shapes(test):
        matmul(kind, *s)
for kind in ("bf16", "block32"):
    matmul(kind, 513 * 256, 8224, 70)
matmul("int8", 513 * 128, 16448, 70)
matmul("int8", 40, 16448, 70)
for mode, h, ffn, seq in T.PREFILL_SHAPES:
    m = T.prefill_model(E, mode, h, ffn, seq)
    c = m.new_llama_kv_cache(seq)
    launches()
    m.prefill([c], np.zeros((1, seq), np.int64))
    record()
    c.free()
    m.free()
every = [k.group() for k in map(KERNEL.search, F.fake_kernels().decode().split()) if k]
print(json.dumps([every, sorted(seen)]))
"""


def test_every_tile_is_reached(fake_hip):
    every, seen = json.loads(fake_hip(RUN).splitlines()[-1])
    seen = {tuple(x) for x in seen}
    missing = []
    for k in every:
        epi = int(k.split("ILi")[1][0])
        staged = k.startswith("k_gemmI")
        if epi and (staged or k.startswith(f"k_gemm_ringILi{epi}ELb0ELb0E")):
            continue  # a model with planes beyond 2 GiB, or k beyond the digit kernel's (which prefill refuses)
        big = "ILi128ELi256E" in k or "ELi128ELi256E" in k
        if (k, False) not in seen and not (epi and (k, True) in seen):
            missing.append(k)
        if epi == 0 and not staged and not big and (k, True) not in seen:
            missing.append(k + " with k splits")
    assert not missing, missing
