"""The dense steps of the Rayleigh-Ritz step at the sizes where their kernels
change (one, two and four rows of a column per lane, the matrix in LDS or one
launch per round, odd n with a dummy index, the one-workgroup solves) against
scipy's generalised eigenproblem: Ritz values to 1e-11 of the spectral scale,
vectors orthonormal to 1e-12, residuals of the rotated pairs to 1e-10."""

import numpy as np
import pytest
import scipy.linalg as sla

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 2, 3, 63, 64, 65, 95, 96, 97, 128, 129, 140, 141, 256, 257])
def test_rayleigh_ritz_sizes(nb):
    import torch

    from cpw2000_amd import hk_psi as hk

    m = 300
    rng = np.random.default_rng(nb)
    a = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))
    a = 0.5 * (a + a.conj().T)
    x = rng.standard_normal((m, nb)) + 1j * rng.standard_normal((m, nb))
    if nb > 40:  # a basis of condition about 100 at every size
        q = np.linalg.qr(x)[0]
        x = q * np.geomspace(1.0, 1e-2, nb)
    hx = a @ x
    h = x.conj().T @ hx
    ref = sla.eigh(0.5 * (h + h.conj().T), x.conj().T @ x, eigvals_only=True)
    psi = torch.from_numpy(np.ascontiguousarray(x.T)).cuda()
    hpsi = torch.from_numpy(np.ascontiguousarray(hx.T)).cuda()
    eig, res = hk.rayleigh_ritz(psi, hpsi)
    assert np.abs(eig - ref).max() < 1e-11 * np.abs(ref).max()
    y, hy = psi.cpu().numpy().T, hpsi.cpu().numpy().T
    assert np.abs(y.conj().T @ y - np.eye(nb)).max() < 1e-12
    assert np.linalg.norm(a @ y - hy) < 1e-11 * np.linalg.norm(hy)
    r = np.sum(np.abs(hy - y * eig) ** 2, axis=0)
    assert np.allclose(res, r, rtol=1e-10, atol=1e-18 * np.abs(ref).max() ** 2)
