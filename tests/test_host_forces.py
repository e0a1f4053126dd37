"""A forces call that fails after its uploads have begun returns only once nothing
reads the caller's arrays any more (on the CPU, against a stand-in for the HIP runtime).
The 128^3 mesh of the 2-atom cell: its density planes do not fit."""

from tests.fake_runtime import run


def test_failed_forces_leave_no_copy_behind():
    out = run("""
d, p = small(kmax_override=[63] * 3)
m, nb = d["mtxd"], 2
f = lambda a: np.ascontiguousarray(a, float)
i = lambda a: np.ascontiguousarray(a, np.int32)
psi = device_array(16 * m * nb)
occ, rat, avec = f(np.ones(nb)), f(np.zeros((2, 3))), f(np.eye(3) * 10.26)
qv, species, fq = i([[1, 0, 0], [0, 1, 0]]), i([0, 0]), f(np.ones(2))
patom, force, enl = i(np.zeros(d["nanl"])), f(np.zeros((2, 3))), f(np.zeros(1))
ptr = lambda a: C.c_void_p(a.ctypes.data)
fake.fake_clear()
rc = hk.lib().cpwgpu_plan_forces(p._h, nb, psi, m, ptr(occ), 2, ptr(rat), ptr(avec), ptr(patom), 2, ptr(qv), 1,
                                 ptr(species), ptr(fq), ptr(force), ptr(enl))
assert rc != 0
seen = log()
assert "copy in" in seen
last = max(k for k, e in enumerate(seen) if e == "copy in")
print("stream sync" in seen[last:])
""")
    assert out.strip() == "True"
