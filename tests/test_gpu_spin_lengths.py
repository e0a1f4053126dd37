"""Two-component H|psi> (nsp = 4) on every specialised mesh length, against the spinor
oracle: the register plane kernel has a block of its own per length in FP64 and another
shape for a box beyond N/4; boxes that just fill N/4 and just exceed it, odd numbers of
band pairs, few and many projectors.  FP64 relative 2-norm error <= 1e-12, FP32-mixed
<= 2e-6.  Where the two sub-planes of FP64 do not fit in LDS the call is refused."""

import numpy as np
import pytest

from oracle import spin
from tests.conftest import rel
from tests.test_gpu_lengths import TOL32, TOL64, _inputs

pytestmark = pytest.mark.gpu

# (n1, n2, n3), largest |k| per direction, bands, projectors, FP64 fits
CASES = [
    ((24, 24, 24), (6, 6, 6), 1, 3, True),
    ((24, 24, 24), (8, 7, 6), 3, 3, True),      # beyond N/4
    ((48, 48, 24), (12, 11, 5), 3, 3, True),
    ((48, 48, 24), (13, 12, 6), 2, 40, True),
    ((64, 64, 24), (16, 16, 6), 1, 3, True),
    ((64, 64, 24), (16, 17, 5), 3, 3, True),
    ((72, 72, 24), (17, 18, 6), 5, 3, True),
    ((72, 72, 24), (19, 18, 6), 1, 3, True),
    ((80, 80, 24), (20, 20, 6), 3, 3, True),
    ((80, 80, 24), (21, 20, 6), 2, 3, True),
    ((96, 96, 24), (24, 24, 6), 1, 3, True),
    ((96, 96, 24), (25, 24, 6), 1, 3, False),
    ((128, 128, 24), (31, 30, 6), 1, 3, False),
]


@pytest.mark.parametrize("n,kd,nb,nanl,fits64", CASES, ids=["x".join(map(str, c[0])) + f"-{c[1][0]}-{c[2]}" for c in CASES])
def test_spin_planes_match_oracle(n, kd, nb, nanl, fits64):
    import torch

    from cpw2000_amd import hk_psi as hk

    d = _inputs(n, kd, nb, nanl)
    m, ntot = d["mtxd"], n[0] * n[1] * n[2]
    rng = np.random.default_rng(m + nb)
    v = np.zeros((d["mxdscr"], 4), order="F")
    v[:ntot] = rng.standard_normal((ntot, 4))
    c = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    beta = np.asfortranarray(c(2 * m, nanl) / np.sqrt(2 * m))
    x = np.asfortranarray(c(2 * m, nb) / np.sqrt(2 * m))
    strength = rng.standard_normal(nanl)
    want = spin.hk_psi_spin(d, x, v, 4, beta, strength, nanl)
    plan = hk.Plan.from_inputs(d, projectors=False)
    plan.set_potential_spin(v, 4)
    plan.set_projectors_spin(beta, strength, nanl)
    xt = torch.from_numpy(np.ascontiguousarray(x.T)).to("cuda")
    for prec, tol in ((hk.PREC_FP64, TOL64), (hk.PREC_FP32, TOL32)):
        ht = torch.full_like(xt, float("nan"))
        if prec == hk.PREC_FP64 and not fits64:
            with pytest.raises(hk.CpwGpuError):
                plan.apply_spin(xt, ht, prec)
            continue
        plan.apply_spin(xt, ht, prec)
        torch.cuda.synchronize()
        assert rel(ht.cpu().numpy().T, want) < tol, (n, prec)
    plan.close()
