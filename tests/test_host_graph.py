"""Which k-points of a graph are launched together, on the CPU against a stand-in for
the HIP runtime: those that take the same kernels and share nothing, in groups of at
most 64; not those of one plan, not a product that is another's input, not those on
two streams or with a kernel that has no batched form."""

from tests.fake_runtime import run

PRELUDE = """
L = hk.lib()

def points(cfgs):
    ds = [small(**kw) for kw in cfgs]
    return [p for _, p in ds], [d["mtxd"] for d, _ in ds]

def graph(plans, ms, nbs, psi=None, hpsi=None, prec=0):
    n = len(plans)
    psi = psi or [device_array(16 * m * max(b, 1)).value for m, b in zip(ms, nbs)]
    hpsi = hpsi or [device_array(16 * m * max(b, 1)).value for m, b in zip(ms, nbs)]
    h = C.c_void_p()
    lds = (C.c_long * n)(*ms)
    hk._check(L.cpwgpu_graph_create(C.byref(h), n, (C.c_void_p * n)(*[p._h.value for p in plans]), (C.c_int * n)(*nbs),
                                    (C.c_void_p * n)(*psi), lds, (C.c_void_p * n)(*hpsi), lds, prec))
    out = (C.c_int * 3)()
    hk._check(L.cpwgpu_graph_info(h, out))
    print(*out)
    L.cpwgpu_graph_destroy(h)
    return psi, hpsi

ks = [dict(kpt=k) for k in ((0, 0, 0), (0.1, 0.2, -0.15), (0.25, -0.25, 0.125), (0.3, 0.1, 0.2))]
"""


def _infos(body):
    return [tuple(int(v) for v in line.split()) for line in run(PRELUDE + body).strip().split("\n")]


def test_groups():
    got = _infos("""
plans, ms = points(ks + [dict(kmax_override=[23] * 3)] * 2)
for prec in (0, 1):
    graph(plans, ms, [16, 16, 16, 16, 16, 16], prec=prec)   # two meshes
    graph(plans, ms, [16, 16, 0, 16, 16, 0], prec=prec)     # without bands
many, mm = points([{}] * 70)
graph(many, mm, [2] * 70)
""")
    assert got == [(6, 2, 6), (6, 1, 3)] * 2 + [(70, 2, 70)]


def test_not_grouped():
    got = _infos("""
plans, ms = points(ks[:1] * 2)
a, b = plans
x, y, z = (device_array(16 * ms[0] * 8).value for _ in range(3))
graph([a, b], ms, [8, 8], [x, y], [y, z])     # one's product is the other's input
graph([a, a], ms, [8, 8])                     # one plan twice
graph([a, b], ms, [8, 8], None, [y, y])       # one output
b.set_variant(0, hk.TUNE_SCHED, 1)
graph([a, b], ms, [8, 8])                     # two streams
b.set_variant(0, hk.TUNE_SCHED, -1)
a.set_variant(0, hk.TUNE_PLANE, 0), b.set_variant(0, hk.TUNE_PLANE, 0)
graph([a, b], ms, [8, 8])                     # a kernel without a batched form
a.set_variant(0, hk.TUNE_PLANE, -1), b.set_variant(0, hk.TUNE_PLANE, -1)
graph([a, b], ms, [8, 8])
""")
    assert got == [(2, 0, 0)] * 5 + [(2, 1, 2)]
