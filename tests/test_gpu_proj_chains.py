"""Accuracy of <beta|psi> with the library's own choice of projection kernel and
slices: no further from the sum in extended precision than the LDS-staged kernel
(number 0) cut into 256 blocks, whose chains of additions the choice is to respect.
With V = 0, no kinetic term and orthonormal projectors of strength 1, beta^H (H psi -
beta c) is the error of c = <beta|psi> (the back-projection's rounding is averaged over
the plane waves).  A rms over 640 to 4,096 complex values is known to 3% and better;
10% are allowed.  (Chains 3 to 7 times as long: 1.4 to 2.1 times the error.)"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(3000, 32, 20), (7550, 64, 64)]  # plane waves, projectors, bands


def _plan(hk, m, nanl, rng):
    k = 13
    g = np.stack(np.meshgrid(*[np.arange(-k, k + 1)] * 3, indexing="ij"), -1).reshape(-1, 3)
    g = g[np.argsort((g ** 2).sum(1), kind="stable")][:m]
    n = 54
    plan = hk.Plan(m, m, np.asfortranarray(g.T.astype(np.int32)), np.zeros(m), np.arange(1, m + 1, dtype=np.int32),
                   np.array([26, 26, 26, n, n, n, n], np.int32))
    plan.set_potential(np.zeros(8 * n ** 3))
    beta = np.linalg.qr(rng.standard_normal((m, nanl)) + 1j * rng.standard_normal((m, nanl)))[0]
    plan.set_projectors(np.asfortranarray(beta), np.ones(nanl))
    return plan, beta


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "fp32mixed"])
@pytest.mark.parametrize("m,nanl,nb", SIZES)
def test_default_split_is_as_accurate_as_256_blocks(m, nanl, nb, prec):
    import torch

    from cpw2000_amd import hk_psi as hk

    rng = np.random.default_rng(m + nb)
    plan, beta = _plan(hk, m, nanl, rng)
    psi = rng.standard_normal((nb, m)) + 1j * rng.standard_normal((nb, m))
    psi /= np.linalg.norm(psi, axis=1)[:, None]
    wide = np.clongdouble if prec == 0 else np.complex128
    b = beta.astype(wide)
    want = b @ (b.conj().T @ psi.T.astype(wide))
    x = torch.from_numpy(psi).to("cuda")

    def error():
        h = torch.full_like(x, float("nan"))
        plan.apply(x, h, prec)
        torch.cuda.synchronize()
        d = b.conj().T @ (h.cpu().numpy().T.astype(wide) - want)
        return float(np.sqrt((np.abs(d) ** 2).mean()))

    chosen = error()
    plan.set_variant(prec, hk.TUNE_PROJ, 0)
    plan.set_variant(prec, hk.TUNE_SPLITK, 256)
    ref = error()
    plan.close()
    assert chosen <= 1.1 * ref, (chosen, ref)
