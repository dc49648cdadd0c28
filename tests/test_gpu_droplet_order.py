"""Droplet rows handed to the library in any order: the order is no part of
the result.

* RK4 sorts its rows by bin; the deposit's fixed-point sums do not depend on
  the order, so permuted rows give the same bits, row by row.
"""
import numpy as np
import pytest

from helpers import inputs
from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


def _t(x, dev, dtype):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev).to(dtype)


def _population(dns, cfg, rows):
    from lucky_droplets_amd.particles import MPI_particles
    return MPI_particles(None, cfg.L, cfg.N, rows.shape[0], cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop, cfg.M0,
                         dns=dns, coord=rows)


@pytest.mark.parametrize("N,prec,npart,speed", [(16, "f64", 1, 1.0), (32, "f32", 777, 1.0), (32, "f64", 5001, 1.0),
                                                (32, "f32", 901, 60.0), (64, "f32", 20011, 1.0)])
def test_rk4_row_order_keeps_the_bits(gpu, N, prec, npart, speed):
    """speed 60: most droplets leave their bin's window within the step (fallback deposit)."""
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    cfg = Config(N=N, precision=prec, nu=0.02, nshells=2, profile="k4", n_particles=npart,
                 st_dist=("uniform", 0.05, 1.0), gravity=True)
    uk, n, coord, _ = inputs(cfg, seed=3, n_noise=0.2)
    coord[:, 3:6] *= speed
    perm = np.random.default_rng(4).permutation(npart)
    out = []
    for rows in (coord, coord[perm]):
        d = ForcedDNS(cfg)
        stb = _population(d, cfg, rows)
        r, u1, n1 = d.RK4(0.0, 0.01, stb, _t(uk, gpu, d.cdtype), _t(n, gpu, d.rdtype))
        out.append((r.cpu().numpy(), u1.cpu().numpy(), n1.cpu().numpy()))
        d.close()
    assert np.isfinite(out[0][0]).all() and np.isfinite(out[0][2]).all()
    assert np.array_equal(out[0][0][perm], out[1][0])
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])
