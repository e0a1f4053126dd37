"""The kernel choice that a plan reports is the one that runs: every value read with
get_variant and set on a second plan of the same k-point gives the product bit for bit,
whether the choice was left to the library or made by the tuner.  Band counts on both
sides of the GEMM tiles' widths, meshes on both sides of the lengths where the
column kernels change."""

import numpy as np
import pytest

from cpw2000_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hk():
    import torch

    from cpw2000_amd import hk_psi

    assert torch.cuda.is_available()
    return hk_psi


def _copy_choice(hk, src, dst, prec):
    for what in (hk.TUNE_PLANE, hk.TUNE_SPLITK, hk.TUNE_PROJ, hk.TUNE_BACK, hk.TUNE_KIN, hk.TUNE_SPIN, hk.TUNE_COL,
                 hk.TUNE_SCHED):
        dst.set_variant(prec, what, src.get_variant(prec, what))


def _bands(d, nb):
    import torch

    p = torch.from_numpy(np.ascontiguousarray(d["psi"][: d["mtxd"]].T)).to("cuda")
    return p[torch.arange(nb) % p.shape[0]].contiguous()


def _same_product(hk, a, b, x, prec):
    import torch

    ha, hb = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    a.apply(x, ha, prec)
    b.apply(x, hb, prec)
    torch.cuda.synchronize()
    assert torch.equal(ha, hb)


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "fp32mixed"])
@pytest.mark.parametrize("cfg,kmax", [(0, None), (0, 31), (1, None)])
def test_defaults_read_and_set(hk, cfg, kmax, prec):
    d = synth.make_config(cfg, nbands=8, **({"kmax_override": [kmax] * 3} if kmax else {}))
    a, b = hk.Plan.from_inputs(d), hk.Plan.from_inputs(d)
    _copy_choice(hk, a, b, prec)
    for nb in (3, 16, 40, 72, 100):
        _same_product(hk, a, b, _bands(d, nb), prec)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "fp32mixed"])
@pytest.mark.parametrize("nb", [16, 72])
def test_tuned_choice_copied(hk, nb, prec):
    import torch

    d = synth.make_config(1, nbands=8)
    a, b = hk.Plan.from_inputs(d), hk.Plan.from_inputs(d)
    x = _bands(d, nb)
    h = torch.zeros_like(x)
    choice = a.tune(x, h, prec)
    for what, key in ((hk.TUNE_PLANE, "plane"), (hk.TUNE_PROJ, "proj"), (hk.TUNE_BACK, "back"),
                      (hk.TUNE_SPLITK, "splitk"), (hk.TUNE_KIN, "kin"), (hk.TUNE_COL, "col"), (hk.TUNE_SCHED, "sched")):
        b.set_variant(prec, what, choice[key])
    _same_product(hk, a, b, x, prec)
    hb = torch.zeros_like(x)
    b.apply(x, hb, prec)
    torch.cuda.synchronize()
    assert torch.equal(h, hb)   # the tuner left the product of its choice
    a.close()
    b.close()
