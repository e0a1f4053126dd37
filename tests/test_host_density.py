"""A density call hands its occupations over on the caller's stream (on the CPU,
against a stand-in for the HIP runtime): no copy of its own beside the kernels of the
call before it, which may still read theirs."""

from tests.fake_runtime import run


def test_occupations_go_in_stream_order():
    out = run("""
d, p = small()
m, nb = d["mtxd"], 300
x, rho = device_array(16 * m * nb), device_array(8 * 24 ** 3)
occ = np.ones(nb)
for _ in range(2):
    fake.fake_clear()
    hk._check(hk.lib().cpwgpu_plan_density(p._h, nb, x, m, C.c_void_p(occ.ctypes.data), rho, None))
    seen = log()
    print(seen.count("copy in"), sum("k_put_occ" in e for e in seen))
""")
    assert out.split() == ["0", "2", "0", "2"]
