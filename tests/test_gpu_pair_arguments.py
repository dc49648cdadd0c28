"""Arguments that the pair statistics refuse."""
import numpy as np
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbins,error", [(8.0, TypeError), (8.5, TypeError), (0, RuntimeError), (513, RuntimeError)])
def test_bin_counts_that_are_refused(gpu, nbins, error):
    from lucky_droplets_amd.dns import ForcedDNS
    from lucky_droplets_amd.particles import MPI_particles
    cfg = Config(N=16, precision="f64", nu=0.02, n_particles=4)
    d = ForcedDNS(cfg)
    stb = MPI_particles(None, cfg.L, cfg.N, 4, cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop, cfg.M0, dns=d,
                        coord=np.random.default_rng(0).uniform(0, 1, (4, 7)))
    with pytest.raises(error):
        stb.pair_statistics(0.1, nbins)
    assert stb.pair_statistics(0.1, 8)["counts"].shape == (8,)
    d.close()
