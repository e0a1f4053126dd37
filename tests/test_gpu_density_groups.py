"""Density planes and forces at the edges of their groups: band counts around
the group sizes of the density pass (one band, one more than a group, many), the
lengths with a shape of their own (80 and 96 with the box inside N/4), a box
beyond N/4 (the shapes that take any box) and 108 (the LDS kernel); forces with
band and projector counts that the MFMA tiles (32 projectors, chunks of 8 bands)
do not divide.  Tolerances: 1e-12 of the largest density (FP64 sums of at most a
few hundred terms), 1e-9 Ha/bohr for forces as in test_gpu_forces.py."""

import numpy as np
import pytest

from cpw2000_amd import synth
from tests.test_gpu_density import _numpy_density

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hk():
    import torch

    from cpw2000_amd import hk_psi

    assert torch.cuda.is_available()
    return hk_psi


def _dev(d, nb):
    import torch

    return torch.from_numpy(np.ascontiguousarray(d["psi"][: d["mtxd"], :nb].T)).to("cuda")


@pytest.mark.parametrize("cfg,nb,kmax", [(0, 1, None), (0, 70, None), (1, 1, None), (1, 14, None), (1, 9, 23),
                                         (4, 3, None), (0, 13, 39), (0, 11, 47), (0, 5, 53)])
def test_density_band_groups(hk, cfg, nb, kmax):
    import torch

    d = synth.make_config(cfg, nbands=nb, kmax_override=None if kmax is None else [kmax] * 3)
    plan = hk.Plan.from_inputs(d, projectors=False)
    occ = np.linspace(2.0, 0.25, nb)
    rho = plan.density(_dev(d, nb), occ)
    torch.cuda.synchronize()
    n = [int(x) for x in d["kmscr"][3:6]]
    ref = _numpy_density(d, d["psi"][:, :nb], occ)
    got = rho.cpu().numpy().reshape(n[2], n[1], n[0])
    plan.close()
    assert np.abs(got - ref).max() < 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("cfg,nb,kmax", [("si2f", 1, None), ("si2f", 9, None), ("si2f", 19, 39), ("si2f", 4, 53),
                                         (4, 5, None)])
def test_forces_ragged_bands(hk, cfg, nb, kmax):
    from oracle import forces as Fo

    d = synth.make_config(cfg, nbands=nb, kmax_override=None if kmax is None else [kmax] * 3)
    plan = hk.Plan.from_inputs(d)
    f, enl = plan.forces(_dev(d, nb), d["rat"], d["avec"], d["proj_atom"], d["floc_q"], d["floc_f"], d["species"])
    plan.close()
    fo, enlo = Fo.forces(d, d["psi"][:, :nb])
    assert np.abs(f - fo).max() < 1e-9
    assert abs(enl - enlo) < 1e-10 * max(1.0, abs(enlo))
