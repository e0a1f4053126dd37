"""Accuracy of the eigenpairs of the LDS subspace eigensolver, seen through the
locally optimal block iteration: each step multiplies the vectors by the eigenvectors
of its subspace, so their departures from orthonormality add up over the steps.  One
step contributes a few roundings for the eigenvectors, the products and the new
directions, together below 16 of 2.2e-16, of either sign: 16 eps sqrt(steps) after all
of them.  (Eigenvectors that are only the product of the sweeps' rotations carry 60
eps and more per step.)  Sums in extended precision on the host.  Subspaces of 24 to 72
and of 42 to 126 columns."""

import numpy as np
import pytest

from cpw2000_amd import synth
from tests.test_gpu_ditsp import EPS, _bufs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg,neig,nvec", [(0, 16, 24), (1, 34, 42)])
@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "fp32mixed"])
def test_block_iteration_keeps_vectors_orthonormal(cfg, neig, nvec, prec):
    import torch

    from cpw2000_amd import hk_psi as hk

    assert torch.cuda.is_available()
    d = synth.make_config(cfg, nbands=1)
    plan = hk.Plan.from_inputs(d)
    psi, hpsi = _bufs(torch, neig, d["mtxd"])
    hk.set_ditsp_method(hk.DITSP_BLOCK)
    try:
        _, ifail, st = plan.ditsp(psi, hpsi, prec=prec, icmax=150, epspsi=EPS)
    finally:
        hk.set_ditsp_method(hk.DITSP_CHEB)
        plan.close()
    assert ifail == 0 and st["nvec"] == nvec, st
    x = psi.cpu().numpy().astype(np.clongdouble)
    off = float(np.abs(x.conj() @ x.T - np.eye(neig)).max())
    assert off < 16 * np.finfo(float).eps * np.sqrt(st["iters"]), (off, st)
