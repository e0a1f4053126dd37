"""The threaded copies of large host matrices, on the CPU against a stand-in for the
HIP runtime: another device after the first large copy, the caller's current device,
pinned memory that is not to be had at first, and the contents.  (2-atom cell, 700
projectors: a matrix of 4.6 MB.)"""

from tests.fake_runtime import run


def test_another_device_after_a_large_copy():
    run("""
fake.fake_devices(2)
L = hk.lib()
hk._check(L.cpwgpu_init(0))
small(700)
hk._check(L.cpwgpu_init(1))
small(700)
""")


def test_current_device_of_the_caller_stays():
    run("""
fake.fake_devices(2)
hk._check(hk.lib().cpwgpu_init(0))
d, p = small()
assert fake.hipSetDevice(1) == 0
big, dev = small(700, seed=1)[0], C.c_int()
p.set_projectors(big["anlga"], big["xnlkb"], 700)
fake.hipGetDevice(C.byref(dev))
assert dev.value == 1, dev.value
""")


def test_pinned_memory_that_comes_later():
    out = run("""
print(hk.host_copy_lanes())
d, p = small()
big = small(700, seed=1)[0]
have = hk.host_copy_lanes()
hk._check(hk.lib().cpwgpu_finalize())
_, p = small()
for refused in (100, 3, 0):   # allocations that fail: all, all but a lane's first, none
    fake.fake_fail_host_malloc(refused)
    p.set_projectors(big["anlga"], big["xnlkb"], 700)
    print(hk.host_copy_lanes())
    fake.fake_fail_host_malloc(0)
print(have)
""").split()
    none, refused, few, later, full = (int(v) for v in out)
    assert none == 0 and refused == 0 and full > 0
    assert few == 0 and later == full
