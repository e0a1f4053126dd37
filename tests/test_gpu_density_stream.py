"""Densities that follow each other on one stream without a wait, with other
occupations each: every result is that of the call alone.  More bands than one block of
kernel arguments holds (256)."""

import numpy as np
import pytest

from cpw2000_amd import synth

pytestmark = pytest.mark.gpu


def test_calls_in_a_row_keep_their_occupations():
    import torch

    from cpw2000_amd import hk_psi as hk

    d = synth.make_config(1, nbands=8)
    plan = hk.Plan.from_inputs(d, projectors=False)
    x = torch.from_numpy(np.ascontiguousarray(d["psi"][: d["mtxd"]].T)).to("cuda")
    x = x[torch.arange(300) % 8].contiguous()
    rng = np.random.default_rng(3)
    occs = [rng.uniform(0.0, 2.0, 300) for _ in range(4)]
    alone = []
    for o in occs:
        alone.append(plan.density(x, o))
        torch.cuda.synchronize()
    row = [plan.density(x, o) for o in occs]
    torch.cuda.synchronize()
    for a, b in zip(alone, row):
        assert torch.equal(a, b)
    # and they are the occupations that were given: the sum over the mesh is linear in them
    one = [float(plan.density(x[:8], np.eye(8)[j]).sum()) for j in range(8)]
    for o, a in zip(occs, alone):
        want = sum(w * one[j % 8] for j, w in enumerate(o))
        assert abs(float(a.sum()) - want) < 1e-11 * want
    plan.close()
