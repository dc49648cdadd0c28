"""Setting and reading an ensemble's state moves every realization in one
launch: fields, and rows at odd counts, come back as they went in, each
realization its own."""
import numpy as np
import pytest

from helpers import inputs
from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,npart", [(2, 1), (3, 257), (5, 33)])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_state_comes_back(gpu, prec, B, npart):
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    cfg = Config(N=16, precision=prec, nu=0.05, nshells=2, profile="k4", n_particles=npart)
    d = ForcedDNS(cfg, batch=B)
    parts = [inputs(cfg, seed=40 + b) for b in range(B)]

    uk, n, rows = (torch.from_numpy(np.stack([np.ascontiguousarray(p[k]) for p in parts])).to(gpu).to(t)
                   for k, t in ((0, d.cdtype), (1, d.rdtype), (2, torch.float64)))
    back = [torch.zeros_like(x) for x in (uk, n, rows)]
    d.set_state(uk, n, rows)
    d.get_state(*back)
    torch.cuda.synchronize()
    assert torch.equal(back[0], uk) and torch.equal(back[1], n)
    assert torch.equal(back[2][..., :3], rows[..., :3])
    vm = rows[..., 3:] if prec == "f64" else rows[..., 3:].float().double()
    assert torch.equal(back[2][..., 3:], vm)
    d.close()
