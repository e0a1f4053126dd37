"""Small k-points of one graph launched together: every replay equals the eager
products bit for bit, for uneven plane-wave and band counts (a k-point without
bands among them), k-points of two meshes, and more than one group; k-points that
depend on each other (one plan twice, the product of one the input of the next)
keep their order."""

import numpy as np
import pytest

from cpw2000_amd import synth

pytestmark = pytest.mark.gpu

KPTS = [(0.0, 0.0, 0.0), (0.1, 0.2, -0.15), (0.25, -0.25, 0.125), (0.3, 0.1, 0.2), (0.05, 0.0, 0.4)]


@pytest.fixture(scope="module")
def hk():
    import torch

    from cpw2000_amd import hk_psi

    assert torch.cuda.is_available()
    return hk_psi


def _psi(d, nb):
    import torch

    p = torch.from_numpy(np.ascontiguousarray(d["psi"][: d["mtxd"]].T)).to("cuda")
    return p[torch.arange(nb) % p.shape[0]].contiguous()


def _replays(hk, plans, psis, prec):
    import torch

    want = []
    for p, x in zip(plans, psis):
        h = torch.zeros_like(x)
        if x.shape[0]:
            p.apply(x, h, prec)
        want.append(h)
    torch.cuda.synchronize()
    outs = [torch.zeros_like(x) for x in psis]
    g = hk.Graph(plans, psis, outs, prec)
    for rep in range(3):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        g.launch()
        torch.cuda.synchronize()
        for k, (w, o) in enumerate(zip(want, outs)):
            assert torch.equal(w, o), (rep, k)
        plans[0].apply(psis[0], torch.zeros_like(psis[0]), prec)
        torch.cuda.synchronize()
    g.close()


@pytest.mark.parametrize("prec", [0, 1])
def test_uneven_points_and_two_meshes(hk, prec):
    ds = [synth.make_config(0, kpt=k) for k in KPTS] + [synth.make_config(0, kpt=KPTS[1], kmax_override=[23] * 3)] * 2
    plans = [hk.Plan.from_inputs(d) for d in ds]
    psis = [_psi(d, nb) for d, nb in zip(ds, (16, 1, 0, 37, 16, 5, 80))]
    _replays(hk, plans, psis, prec)
    # without projectors: fewer steps
    bare = [hk.Plan.from_inputs(d, projectors=False) for d in ds[:2]]
    _replays(hk, bare + plans[2:4], psis[:4], prec)
    for p in plans + bare:
        p.close()


def test_more_points_than_one_group(hk):
    d = synth.make_config(0)
    plans = [hk.Plan.from_inputs(d) for _ in range(70)]
    _replays(hk, plans, [_psi(d, 1 + k % 3) for k in range(70)], hk.PREC_FP64)
    for p in plans:
        p.close()


def test_dependent_points_keep_their_order(hk):
    import torch

    d = synth.make_config(0)
    a, b = hk.Plan.from_inputs(d), hk.Plan.from_inputs(d)
    x = _psi(d, 8)
    y, z = torch.zeros_like(x), torch.zeros_like(x)
    a.apply(x, y, hk.PREC_FP64)
    b.apply(y, z, hk.PREC_FP64)
    torch.cuda.synchronize()
    y2, z2 = torch.zeros_like(x), torch.zeros_like(x)
    g = hk.Graph([a, b], [x, y2], [y2, z2])
    g2 = hk.Graph([a, a], [x, y], [torch.zeros_like(x), torch.zeros_like(x)])
    for _ in range(2):
        y2.zero_(), z2.zero_()
        torch.cuda.synchronize()
        g.launch()
        g2.launch()
        torch.cuda.synchronize()
        assert torch.equal(y2, y) and torch.equal(z2, z)
        assert torch.equal(g2._keep[2][0], y) and torch.equal(g2._keep[2][1], z)
    g.close()
    g2.close()
    a.close()
    b.close()
