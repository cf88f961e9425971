"""The storage pool's bound, its sizes and what it gives back (host logic, on a
runtime without a device).  Sizes in f32 values."""


def test_cache_is_bounded_and_keeps_the_last_freed(fake_hip):
    fake_hip("""
small = [B.zeros(1000 + 100 * i) for i in range(20)]
big = [B.zeros(1 << 27) for _ in range(6)]  # 512 MB each
live = F.fake_used()
for s in big: s.free()
for s in small: s.free()
assert F.fake_used() <= 2 << 30 and F.fake_used() > 1 << 30
n = F.fake_mallocs()
again = [B.zeros(1000 + 100 * i) for i in range(20)] + [B.zeros(1 << 27) for _ in range(3)]
assert F.fake_mallocs() == n
from esolearn_amd._lib import call
call("scry_hip_shutdown")
assert F.fake_used() < (3 << 29) + (1 << 20)  # the live storage
""")


def test_cache_full_of_blocks_no_longer_used(fake_hip):
    """They make room for the blocks in use, which then stay."""
    fake_hip("""
old = [B.zeros(75 << 20) for _ in range(6)] + [B.zeros(1000 + i) for i in range(300)]  # 6 x 300 MB
for s in old: s.free()
for step in range(4):
    n = F.fake_mallocs()
    s = [B.zeros(1 << 27) for _ in range(3)]
    for x in s: x.free()
    assert step < 2 or F.fake_mallocs() == n, step
""")


def test_cached_blocks_are_given_back_for_an_allocation(fake_hip):
    fake_hip("""
s = [B.zeros(1 << 26) for _ in range(4)]  # 1 GB
used = F.fake_used()
F.fake_limit(used)
for b in s: b.free()
assert F.fake_used() == used
x = B.zeros(200 << 20)  # 800 MB: only without the cache
assert F.fake_used() < used
""")


def test_large_blocks_have_their_exact_size(fake_hip):
    fake_hip("""
used = F.fake_used()
n = (1 << 28) + 3
x = B.zeros(n)
assert F.fake_used() - used == 4 * n
x.free()
assert F.fake_used() == used
""")


def test_a_size_that_fits_exactly(fake_hip):
    fake_hip("""
n = (1 << 26) + 3  # its class has 32 MB more
F.fake_limit(F.fake_used() + 4 * n)
x = B.zeros(n)
used = F.fake_used()
x.free()
assert F.fake_used() == used - 4 * n  # not kept under a class it is too small for
""")


def test_sizes_beyond_any_device_are_refused(fake_hip):
    fake_hip("""
for n in ((1 << 62) - 1, (1 << 61) + (1 << 60) + 1, 1 << 50):
    try:
        B.zeros(n)
    except E.ScryHipError as e:
        assert e.code == 3
    else:
        raise SystemExit(f"{n} values were accepted")
""")
