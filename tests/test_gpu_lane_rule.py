"""The lanes per droplet of the stage kernel (4 or 8, by counts and sizes;
LD_STAGE_LANES sets them) are no part of the result."""
import numpy as np
import pytest

from helpers import inputs
from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,prec,npart,batch", [(16, "f64", 1, 1), (16, "f32", 683, 1), (32, "f64", 5470, 1),
                                                (32, "f32", 8191, 1), (64, "f32", 40_001, 1), (32, "f32", 1000, 3)])
def test_four_and_eight_lanes_give_the_same_bits(gpu, N, prec, npart, batch, monkeypatch):
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    cfg = Config(N=N, precision=prec, nu=0.05, nshells=2, profile="k4", n_particles=npart,
                 st_dist=("uniform", 0.05, 1.0), gravity=True)
    uk, n, coord, _ = inputs(cfg, seed=11, n_noise=0.2)
    got = []
    for lanes in ("4", "8", "0"):
        monkeypatch.setenv("LD_STAGE_LANES", lanes)
        d = ForcedDNS(cfg, batch=batch)
        t = [torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (uk, n, coord)]
        t = [t[0].to(d.cdtype), t[1].to(d.rdtype), t[2]]
        if batch > 1:
            t = [torch.stack([x * (1 + 0.01 * b) for b in range(batch)]) for x in t]
        d.set_state(*t)
        d.advance(0.01, 2)
        d.get_state(*t)
        got.append([x.cpu().numpy() for x in t])
        d.close()
    assert all(np.isfinite(x).all() for x in got[0])
    for o in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got[0], o))
