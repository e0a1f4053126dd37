"""The diagonalisation at the block sizes where its dense steps change kernels: an
odd and a tiny block, 65 and 128 vectors (two rows per lane, the largest subspace
of the LDS eigensolver), 135 (the library eigensolver with the LDS factor).  The
checks are those of test_gpu_ditsp.py: orthonormal vectors to 1e-12, hpsi against an
independent product, residuals below epspsi; and the lowest eigenvalues agree between
the blocks to 1e-9 Ha (a Ritz value's error is of the order of its residual squared)."""

import numpy as np
import pytest

from cpw2000_amd import synth
from tests.test_gpu_ditsp import EPS, _bufs, _check_pairs

pytestmark = pytest.mark.gpu


def test_blocks_around_the_eigensolver_sizes():
    import torch

    from cpw2000_amd import hk_psi as hk

    assert torch.cuda.is_available()
    d = synth.make_config(1, nbands=1)
    plan = hk.Plan.from_inputs(d)
    low = {}
    for neig in (1, 57, 114, 120):
        psi, hpsi = _bufs(torch, neig, d["mtxd"])
        ei, ifail, st = plan.ditsp(psi, hpsi, prec=hk.PREC_FP32, icmax=100, epspsi=EPS)
        assert ifail == 0, (neig, st)
        _check_pairs(torch, plan, hk, psi, hpsi, ei)
        low[neig] = ei
    plan.close()
    for neig in (1, 57, 114):
        assert np.abs(low[neig] - low[120][:neig]).max() < 1e-9
