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
