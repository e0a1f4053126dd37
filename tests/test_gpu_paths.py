"""The paths that results alone do not tell apart, on the device: k-points of a graph
launched together, a large host matrix copied by threads."""

import numpy as np
import pytest

from cpw2000_amd import synth

pytestmark = pytest.mark.gpu


def test_grouped_points_and_copying_threads():
    import torch

    from cpw2000_amd import hk_psi as hk

    assert torch.cuda.is_available()
    d = synth.make_config(0)
    plans = [hk.Plan.from_inputs(d) for _ in range(6)]
    x = torch.from_numpy(np.ascontiguousarray(d["psi"][: d["mtxd"]].T)).to("cuda")
    g = hk.Graph(plans, [x] * 6, [torch.zeros_like(x) for _ in plans])
    assert g.info() == {"points": 6, "groups": 1, "grouped": 6}
    g.close()
    for p in plans:
        p.close()
    hk.Plan.from_inputs(synth.make_config(1, nbands=1)).close()   # 98 MB of projectors
    assert hk.host_copy_lanes() > 0
