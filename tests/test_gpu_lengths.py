"""H|psi> with the library's own kernel choice on the mesh lengths and boxes
where that choice changes, against the oracle: every length with a pruned
register plane shape, boxes that just fill N/4 and just exceed it, meshes whose
columns are specialised and whose planes are not, and band and projector counts
on both sides of the GEMM tile widths.  FP64 relative 2-norm error <= 1e-12,
FP32-mixed <= 2e-6."""

import numpy as np
import pytest

from tests.conftest import rel

pytestmark = pytest.mark.gpu

TOL64, TOL32 = 1e-12, 2e-6

# (n1, n2, n3), largest |k| per direction, bands, projectors
CASES = [
    ((18, 18, 18), (4, 4, 4), 3, 5),
    ((20, 20, 20), (5, 5, 5), 16, 8),       # box at N/4
    ((32, 32, 32), (8, 8, 8), 5, 33),
    ((36, 36, 36), (8, 9, 8), 33, 32),
    ((36, 36, 36), (12, 9, 9), 3, 5),       # box wider than N/4: generic plane kernel
    ((40, 40, 40), (10, 10, 9), 2, 1),
    ((50, 50, 50), (12, 12, 12), 3, 5),
    ((54, 54, 54), (13, 13, 13), 3, 5),
    ((80, 80, 24), (19, 19, 5), 2, 70),
    ((80, 80, 24), (20, 20, 6), 2, 5),      # box at N/4: wider than the compile-time row stride
    ((96, 96, 24), (24, 23, 6), 2, 5),
    ((100, 100, 18), (25, 24, 4), 2, 5),
    ((108, 108, 20), (27, 26, 5), 2, 5),
    ((128, 128, 24), (31, 32, 5), 1, 5),
    ((32, 32, 128), (7, 7, 31), 4, 300),
    ((72, 72, 36), (17, 17, 9), 65, 130),
    ((36, 50, 50), (8, 12, 12), 3, 5),      # n1 != n2
    ((12, 12, 54), (3, 3, 13), 3, 5),       # generic plane, specialised columns
    ((24, 24, 30), (6, 6, 7), 3, 5),        # specialised plane, generic columns
]


def _inputs(n, kd, nb, nanl):
    """Random plane waves that reach kd in every direction, projectors, V and bands."""
    rng = np.random.default_rng(sum(n) + 7 * nb + nanl)
    g = np.stack([rng.integers(-k, k + 1, 900) for k in kd], 1)
    for j in range(3):
        for s in (-1, 1):
            e = np.zeros(3, int)
            e[j] = s * kd[j]
            g = np.vstack([g, e])
    g = np.unique(g, axis=0)
    rng.shuffle(g)
    m = len(g)
    c = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    ntot = n[0] * n[1] * n[2]
    f = np.asfortranarray
    return dict(mtxd=m, ng=m, mxddim=m, mxdgve=m, mxdanl=max(nanl, 1), nanl=nanl, mxdbnd=nb, mxdscr=8 * ntot,
                kgv=f(g.T.astype(np.int32)), isort=np.arange(1, m + 1, dtype=np.int32),
                ekpg=0.05 * (g ** 2).sum(1).astype(float),
                kmscr=np.array([*((k - 1) // 2 for k in n), *n, n[0]], np.int32),
                vscr=np.concatenate([rng.standard_normal(ntot), np.zeros(7 * ntot)]),
                psi=f(c(m, nb) / np.sqrt(m)), anlga=f(c(m, max(nanl, 1)) / np.sqrt(m)),
                xnlkb=rng.standard_normal(max(nanl, 1)))


@pytest.mark.parametrize("n,kd,nb,nanl", CASES, ids=["x".join(map(str, c[0])) + f"-{c[1][0]}-{c[2]}" for c in CASES])
def test_default_kernels_match_oracle(orc, n, kd, nb, nanl):
    import torch

    from cpw2000_amd import hk_psi as hk

    d = _inputs(n, kd, nb, nanl)
    st, href = orc.orc_hk_psi(d)
    assert st == 0
    plan = hk.Plan.from_inputs(d)
    pt = torch.from_numpy(np.ascontiguousarray(d["psi"].T)).to("cuda")
    for prec, tol in ((hk.PREC_FP64, TOL64), (hk.PREC_FP32, TOL32)):
        ht = torch.full_like(pt, float("nan"))
        plan.apply(pt, ht, prec)
        torch.cuda.synchronize()
        assert rel(ht.cpu().numpy().T, href) < tol, (n, prec)
    plan.close()
