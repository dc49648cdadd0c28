"""The droplet stage's counters and fallback sums across stages, steps and
replays: the fallback slots are deposited by the brick launch, folded into the
deposit by the z pass that reads it, and the counters cleared by the chain's
last kernel, so every stage has to find them clean.  Steps in one call, one
by one and replayed from a graph give the same bits, fast droplets (most in the
fallback) included; a growth rate that is not a number makes the density NaN."""
import numpy as np
import pytest

from helpers import inputs
from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


def _run(gpu, cfg, arrays, h, calls, graph=False):
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    d = ForcedDNS(cfg, graph=graph)
    uk, n, rows = (torch.from_numpy(np.ascontiguousarray(a)).to(gpu) for a in arrays)
    t = [uk.to(d.cdtype), n.to(d.rdtype), rows]
    d.set_state(*t)
    for k in calls:
        d.advance(h, k)
    d.get_state(*t)
    out = [x.cpu().numpy() for x in t]
    d.close()
    return out


@pytest.mark.parametrize("N,prec,npart", [(16, "f32", 33), (32, "f64", 1), (64, "f32", 1500), (64, "f64", 700),
                                          (128, "f32", 5000)])
def test_fast_droplets_over_steps_and_replays(gpu, N, prec, npart):
    cfg = Config(N=N, precision=prec, nu=0.05, nshells=2, profile="k4", n_particles=npart,
                 st_dist=("uniform", 0.05, 1.0), gravity=False)
    uk, n, coord, _ = inputs(cfg, seed=5)
    h = 0.2 / N
    coord[: max(1, 2 * npart // 3), 3:6] *= 30.0           # several bins per stage
    arrays = (uk, n, coord)
    a = _run(gpu, cfg, arrays, h, (4,))
    assert all(np.isfinite(x).all() for x in a)
    for calls, graph in (((1, 1, 1, 1), False), ((2, 2), True)):
        b = _run(gpu, cfg, arrays, h, calls, graph)
        for x, y in zip(a, b):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (calls, graph)


@pytest.mark.parametrize("fast", [False, True])
def test_not_a_number_growth_reaches_the_density(gpu, fast):
    cfg = Config(N=32, precision="f64", nu=0.05, nshells=2, profile="k4", n_particles=50)
    uk, n, coord, _ = inputs(cfg, seed=6)
    coord[7, 6] = np.nan
    if fast:
        coord[:, 3:6] *= 40.0
    out = _run(gpu, cfg, (uk, n, coord), 0.005, (1,))
    assert np.isnan(out[1]).all()
    assert np.isfinite(out[0]).all()
