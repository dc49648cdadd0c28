"""Collision pairs beyond 2^30: the sort's key numbers pass 32 bits."""
import numpy as np
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


def test_more_than_2_to_the_30_pairs(gpu):
    """46342 droplets that all overlap: every (i, j), i < j, once and in order
    (the sort runs over 2^31 keys, 2^30 + 25487 of them pairs)."""
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    from lucky_droplets_amd.particles import MPI_particles
    if torch.cuda.mem_get_info()[0] < 100 << 30:
        pytest.skip("needs 100 GB of device memory")
    n = 46342
    total = n * (n - 1) // 2
    assert total > 1 << 30
    cfg = Config(N=16, precision="f64", nu=0.02, n_particles=n)
    d = ForcedDNS(cfg)
    rows = np.random.default_rng(0).uniform(0, 0.1, (n, 7))
    stb = MPI_particles(None, cfg.L, cfg.N, n, cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop, cfg.M0, dns=d,
                        coord=rows)
    got = stb.collision_pairs(torch.full((n,), 0.2, dtype=torch.float64, device=gpu), max_pairs=total)
    assert got.shape == (total, 2)
    last = -1
    for part in torch.split(got, 1 << 27):
        i, j = part[:, 0], part[:, 1]
        key = i * n + j
        assert bool(((i >= 0) & (i < j) & (j < n)).all())
        # strictly increasing: with the count, every pair once and sorted
        assert int(key[0]) > last and bool((key[1:] > key[:-1]).all())
        last = int(key[-1])
    del got, part, i, j, key
    d.close()
    torch.cuda.empty_cache()
