"""The pair search's cell walk, queue and sort at the sizes where they can go
wrong, against the brute-force specification (bit-exact pairs and counts)."""
import numpy as np
import pytest

from lucky_droplets_amd.config import Config


def test_minimum_image_by_comparison_equals_rounded_quotient():
    """For wrapped positions t = x_j - x_i lies in [-L, L] and rint(t / L) is 1
    above L/2, -1 below -L/2, else 0, to the last bit around L/2."""
    rng = np.random.default_rng(0)
    for L in np.concatenate([[2 * np.pi, 1.0, 3.0, 2.0 - 2.0 ** -52, 1.0 + 2.0 ** -52], rng.uniform(0.1, 50.0, 2000)]):
        h = 0.5 * L
        t = [0.0, L, np.nextafter(L, 0), h]
        for d in (0.0, 2 * L):
            x = h
            for _ in range(4):
                x = np.nextafter(x, d)
                t.append(x)
        t = np.array(t + list(rng.uniform(0, L, 50)))
        t = np.concatenate([t, -t])
        by_compare = np.where(t > h, t - L, np.where(t < -h, t + L, t))
        assert np.array_equal(t - L * np.rint(t / L), by_compare)


def _stb(n, rows, N=32):
    from lucky_droplets_amd.dns import ForcedDNS
    from lucky_droplets_amd.particles import MPI_particles
    cfg = Config(N=N, precision="f64", nu=0.02, n_particles=max(1, n))
    d = ForcedDNS(cfg)
    return d, MPI_particles(None, cfg.L, cfg.N, n, cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop, cfg.M0, dns=d,
                            coord=rows)


def _rows(n, seed, spread=1.0):
    rng = np.random.default_rng(seed)
    L = 2 * np.pi
    rows = rng.uniform(0, L, (n, 7))
    rows[:, :3] = (rows[:, :3] - 0.5 * L) * spread            # a cluster over the box's corner when spread < 1
    rows[:, :3] += L * rng.integers(-2, 3, (n, 3))
    rows[:, 3:6] = rng.standard_normal((n, 3))
    if n > 3:
        rows[1, :3] = rows[0, :3]                             # coincident droplets
        rows[2, :3], rows[3, :3] = (0.0, 0.0, 0.0), (np.pi, 0.0, np.pi)
    return rows


# reach = 2 r: 3 cells per side (r = 1), 4 (0.75), one cell (1.2), many; pair counts on both sides of the 2048-key
# sort chunk and over several chunks
@pytest.mark.gpu
@pytest.mark.parametrize("n,r,spread", [(2, 1.6, 1.0), (64, 1.0, 1.0), (170, 1.0, 1.0), (176, 1.0, 1.0), (260, 1.0, 1.0),
                                        (400, 0.75, 1.0), (300, 1.2, 1.0), (2000, 0.05, 0.2), (3001, 0.02, 1.0)])
def test_pairs_against_brute_force(gpu, n, r, spread):
    import torch
    from oracle import collide
    rows = _rows(n, n, spread)
    rad = np.random.default_rng(n + 1).uniform(0.6 * r, r, n)
    d, stb = _stb(n, rows)
    got = stb.collision_pairs(torch.from_numpy(rad).to(gpu), max_pairs=1 << 18).cpu().numpy()
    assert np.array_equal(got, collide.pairs_bruteforce(rows, rad, 2 * np.pi))
    d.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,rmax,nbins,spread", [(2, 3.0, 1, 1.0), (65, 2.0, 7, 1.0), (700, 1.5, 512, 1.0),
                                                 (1500, 0.3, 33, 0.2), (3000, 0.12, 64, 1.0)])
def test_statistics_against_brute_force(gpu, n, rmax, nbins, spread):
    from oracle import collide
    rows = _rows(n, 10 + n, spread)
    d, stb = _stb(n, rows)
    got = stb.pair_statistics(rmax, nbins)
    c, ws, wn = collide.pair_stats_bruteforce(rows, 2 * np.pi, rmax, nbins)
    assert np.array_equal(got["counts"], c)
    # FP64 sums of at most 10^5 terms in another order
    assert np.allclose(got["wsum"], ws, rtol=1e-11, atol=0) and np.allclose(got["wneg"], wn, rtol=1e-11, atol=0)
    d.close()


@pytest.mark.gpu
def test_growing_and_shrinking_populations(gpu):
    """One context, populations of changing size: the workspaces follow."""
    import torch
    from oracle import collide
    d, _ = _stb(1, _rows(1, 0))
    from lucky_droplets_amd.particles import MPI_particles
    c = d.cfg
    for n in (50, 900, 10, 1000, 3):
        rows = _rows(n, n + 7)
        stb = MPI_particles(None, c.L, c.N, n, c.sts, 0.05, c.g, c.nu_eff, c.tf, c.rhop, c.M0, dns=d, coord=rows)
        rad = np.full(n, 0.15)
        got = stb.collision_pairs(torch.from_numpy(rad).to(gpu)).cpu().numpy()
        assert np.array_equal(got, collide.pairs_bruteforce(rows, rad, 2 * np.pi))
        cnt = stb.pair_statistics(0.4, 9)["counts"]
        assert np.array_equal(cnt, collide.pair_stats_bruteforce(rows, 2 * np.pi, 0.4, 9)[0])
    d.close()
