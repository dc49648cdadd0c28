"""Workspaces of the pair search over a growing population: what earlier sizes
leave behind stays below twice the largest."""
import numpy as np
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


def test_cell_starts_of_a_growing_population(gpu):
    """One cell per droplet: 20^3 .. 120^3 cells, 6.9 MB of starts for the largest (206 MB for all of the sizes)."""
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    from lucky_droplets_amd.particles import MPI_particles
    cfg = Config(N=32, precision="f64", nu=0.02, n_particles=1)
    d = ForcedDNS(cfg)
    top = 120 ** 3
    rows = torch.from_numpy(np.random.default_rng(0).uniform(0, cfg.L, (top, 7))).to(gpu)
    rad = torch.full((top,), 1e-6, dtype=torch.float64, device=gpu)

    rows[:2, :3] = 1.0                     # one pair

    def population(n):
        return MPI_particles(None, cfg.L, cfg.N, n, cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop, cfg.M0, dns=d,
                             coord=rows[:n])

    population(top).coalesce(torch.tensor([[0, 1]], device=gpu))       # the droplets' own arrays, for all of them
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    for nc in range(20, 121):
        assert population(nc ** 3).collision_pairs(rad[: nc ** 3], max_pairs=1 << 10).tolist() == [[0, 1]]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    used = free - torch.cuda.mem_get_info()[0]
    assert used < 3 * 4 * top + (8 << 20), used
    d.close()
