"""The projection and back-projection kernels that the default takes for a number
of bands (16, 32, 48, 64 and 80 bands per block), at counts around their tiles, on
the 64-atom cell and on a small one: FP64 against the plain torch product (1e-13
relative 2-norm, as the variants among each other), FP32-mixed to 2e-6."""

import numpy as np
import pytest

from cpw2000_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg,nanl", [(0, 37), (1, 256)])
def test_default_kernels_by_band_count(cfg, nanl):
    import torch

    from cpw2000_amd import hk_psi as hk

    assert torch.cuda.is_available()
    d = synth.make_config(cfg, nbands=1, with_psi=False)
    m = d["mtxd"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7 + cfg)
    beta = torch.randn(nanl, m, generator=gen, dtype=torch.complex128, device="cuda") / m ** 0.5
    xnl = torch.linspace(-2.0, 2.0, nanl, dtype=torch.float64, device="cuda")
    psi = torch.randn(161, m, generator=gen, dtype=torch.complex128, device="cuda")
    torch.cuda.synchronize()
    plan = hk.Plan.from_inputs(d, projectors=False)
    local = torch.zeros_like(psi)
    plan.apply(psi, local, hk.PREC_FP64)
    torch.cuda.synchronize()
    plan.set_projectors_device(beta, xnl)
    want = local + ((psi @ beta.conj().T) * xnl) @ beta
    for nb in (1, 15, 16, 17, 32, 33, 48, 49, 72, 80, 81, 96, 100, 112, 113, 128, 144, 161):
        for prec, tol in ((hk.PREC_FP64, 1e-13), (hk.PREC_FP32, 2e-6)):
            h = torch.zeros_like(psi[:nb])
            plan.apply(psi[:nb], h, prec)
            torch.cuda.synchronize()
            err = float(torch.linalg.norm(h - want[:nb]) / torch.linalg.norm(want[:nb]))
            assert err < tol, (nb, prec, err)
    plan.close()
