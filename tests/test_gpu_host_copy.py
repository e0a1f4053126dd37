"""The host-array call with matrices large enough for the threaded copies: columns
with and without rows beyond mtxd (which keep their contents), band counts whose last
chunk is short, equal to the device-resident product bit for bit, call after call."""

import numpy as np
import pytest

from cpw2000_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pad", [0, 13])
def test_host_call_equals_resident_product(pad):
    import torch

    from cpw2000_amd import hk_psi as hk

    assert torch.cuda.is_available()
    d = synth.make_config(1, nbands=23, mxddim_pad=pad)
    m = d["mtxd"]
    plan = hk.Plan.from_inputs(d)
    for nb in (23, 11, 5, 23):     # 5 bands: below the threaded copies, the projectors above
        x = torch.from_numpy(np.ascontiguousarray(d["psi"][:m, :nb].T)).to("cuda")
        want = torch.zeros_like(x)
        plan.apply(x, want, hk.PREC_FP64)
        torch.cuda.synchronize()
        h = np.full_like(d["psi"], 7.0, order="F")
        hk.hk_psi_c16_dict(d, hpsi=h, neig=nb)
        assert np.array_equal(h[:m, :nb], want.cpu().numpy().T)
        assert np.all(h[m:] == 7.0) and np.all(h[:, nb:] == 7.0)
    plan.close()
