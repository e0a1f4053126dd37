"""cpwgpu_finalize gives every buffer of the library back (on the CPU, against a
stand-in for the HIP runtime), and the library works again afterwards."""

from tests.fake_runtime import run


def test_finalize_gives_every_buffer_back():
    out = run("""
L = hk.lib()
f = lambda a: np.ascontiguousarray(a, float)
i = lambda a: np.ascontiguousarray(a, np.int32)
ptr = lambda a: C.c_void_p(a.ctypes.data)
for again in range(2):
    d, p = small(700)
    m, nb = d["mtxd"], 100
    x, h = device_array(16 * m * nb), device_array(16 * m * nb)
    for prec in (0, 1):
        hk._check(L.cpwgpu_plan_apply(p._h, nb, x, m, h, m, prec, None))
    rho = device_array(8 * 24 ** 3)
    occ, eig, res = f(np.ones(nb)), f(np.zeros(nb)), f(np.zeros(nb))
    hk._check(L.cpwgpu_plan_density(p._h, nb, x, m, ptr(occ), rho, None))
    rat, avec, force = f(np.zeros((2, 3))), f(np.eye(3) * 10.26), f(np.zeros((2, 3)))
    qv, species, fq, patom = i([[1, 0, 0], [0, 1, 0]]), i([0, 0]), f(np.ones(2)), i(np.zeros(700))
    hk._check(L.cpwgpu_plan_forces(p._h, nb, x, m, ptr(occ), 2, ptr(rat), ptr(avec), ptr(patom), 2, ptr(qv), 1,
                                   ptr(species), ptr(fq), ptr(force), None))
    for n in (40, 100):   # the matrix in LDS, a launch per round
        hk._check(L.cpwgpu_rayleigh_ritz(m, n, x, m, h, m, 1, ptr(eig), ptr(res), None))
    hk.hk_psi_c16_dict(d)
    p.close()
    for a in (x, h, rho):
        fake.hipFree(a)
    hk._check(L.cpwgpu_finalize())
    print(fake.fake_live())
""")
    assert out.split() == ["0", "0"]
