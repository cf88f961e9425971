"""Where the device has no memory left for a workspace the work runs without
it, and an op that fails leaves no output (host logic, on a runtime without a
device)."""
import pytest

OPS = """
A, W = B.zeros(64 * 4096), B.zeros(4096 * 4096)
Q, SC = B.i8_from_vec(np.zeros(4096 * 4096, np.int8)), B.zeros(4096 * 128)
def bf16(m):
    B.set_bf16_mode(True)
    try:
        return B.matmul(B.zeros(m * 4096) if m < 64 else A, W, m, 4096, 4096)
    finally:
        B.set_bf16_mode(False)
op = dict(matmul=lambda m=64: B.matmul(A, W, 64, 4096, 4096),
          few_rows=lambda m=2: B.matmul_strided_batched(A, W, 1, 2, 4096, 4096),
          bias=lambda m=64: B.matmul_bias(A, W, A, 64, 4096, 4096),
          digits=lambda m=64: B.matmul_i8_f32(B.zeros(m * 4096), Q, 1.0, m, 4096, 4096),
          block32=lambda m=64: B.matmul_i8_f32_block32(B.zeros(m * 4096), Q, SC, m, 4096, 4096),
          bf16=lambda m=64: bf16(m))
def split(o):
    launches()
    o()
    names = [l.split()[0] for l in launches()]
    assert any("k_mm_f64" in n or "k_mv_cols" in n or "k_gemm" in n for n in names), names
    return any(f in n for f in ("k_mm_reduce", "k_digits_finish", "k_ring_finish") for n in names)
"""


@pytest.mark.parametrize("op", ["matmul", "few_rows", "bias", "digits", "block32", "bf16"])
def test_no_room_for_partial_sums(fake_hip, op):
    fake_hip(OPS + f"""
op = op[{op!r}]
if {op!r} in ("digits", "block32", "bf16"):
    op(1)  # the weights' packed rows
used = F.fake_used()
F.fake_limit(used + (1 << 20 if {op!r} == "few_rows" else 5 << 20))  # activations and outputs, but no partial sums
assert not split(op)
F.fake_limit(1 << 40)
assert split(op)  # and with room again
""")


@pytest.mark.parametrize("call", ["matmul(A.h, W.h, 64, 4096, 4096, 0, 0", "matmul_bias(A.h, W.h, A.h, 64, 4096, 4096, 0, 0",
                                  "matmul_strided_batched(A.h, W.h, 1, 64, 4096, 4096, 0, 0"])
def test_failed_op_leaves_no_output(fake_hip, call):
    """The launch is refused (here by a grid the runtime does not take)."""
    fake_hip(OPS + f"""
from esolearn_amd._lib import load
out = C.c_void_p()
F.fake_refuse(1)
rc = load().scry_hip_{call}, C.byref(out))
F.fake_refuse(0)
assert rc != 0 and not out.value, (rc, out)
""")
