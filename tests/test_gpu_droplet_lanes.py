"""The droplet stage takes 8 lanes per droplet below one droplet in 6 cells and
4 above: steps on both sides of that line, with droplet counts that leave
partial blocks and wavefronts, against the oracle (forced-dns-sm.py:335-362).
Tolerances as for whole steps: 1e-10 in FP64, 1e-4 in FP32."""
import numpy as np
import pytest

from helpers import by_id, inputs, make_drops_oracle, make_flow_oracle, min_image, relerr
from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-10, "f32": 1e-4}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("N,npart", [(16, 1), (16, 33), (16, 682), (16, 683), (32, 257), (32, 5470)])
def test_steps_on_both_sides_of_the_lane_rule(gpu, N, npart, prec):
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    cfg = Config(N=N, precision=prec, nu=0.05, nshells=2, profile="k4", n_particles=npart,
                 st_dist=("uniform", 0.05, 1.0), gravity=True)
    uk, n, coord, pid = inputs(cfg, seed=31)
    fl = make_flow_oracle(cfg)
    dr = make_drops_oracle(cfg, coord, pid)
    h = 0.01
    uk_r, n_r = uk.copy(), n.copy()
    for _ in range(2):
        uk_r, n_r = fl.step(0.0, h, dr, uk_r, n_r)
    d = ForcedDNS(cfg)
    u, m, c = (torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (uk, n, coord))
    u, m = u.to(d.cdtype), m.to(d.rdtype)
    d.set_state(u, m, c)
    d.advance(h, 2)
    d.get_state(u, m, c)
    torch.cuda.synchronize()
    tol = TOL[prec]
    assert relerr(u.cpu().numpy(), uk_r) < tol
    assert relerr(m.cpu().numpy(), n_r) < tol
    a, b = c.cpu().numpy(), by_id(dr.coord, dr.prtclid)
    assert min_image(a, b, cfg.L) < tol * cfg.L
    assert relerr(a[:, 3:], b[:, 3:]) < tol
    d.close()
