"""Populations that cluster: the same answers, and no serial work in the few
cells, tiles or bricks that hold them.

The time bounds are ratios to a uniform population of the same size: a cluster
whose work ran in one workgroup, or whose droplets all shared a few cells, cost
85 to 100 times as much."""
import numpy as np
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


def _population(N, prec, rows, batch=1):
    from lucky_droplets_amd.dns import ForcedDNS
    from lucky_droplets_amd.particles import MPI_particles
    cfg = Config(N=N, precision=prec, nu=0.02, n_particles=rows.shape[0])
    d = ForcedDNS(cfg)
    return d, MPI_particles(None, cfg.L, cfg.N, rows.shape[0], cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop,
                            cfg.M0, dns=d, coord=rows)


def _rows(n, side, seed=0):
    """n rows in a box of side L * side, off the box's corner."""
    rows = np.random.default_rng(seed).uniform(0, 2 * np.pi, (n, 7))
    rows[:, :3] = rows[:, :3] * side + 1.0
    rows[:, 6] *= 1e-4
    return rows


def _ms(f):
    import torch
    f()
    t = []
    for _ in range(3):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        f()
        b.record()
        b.synchronize()
        t.append(a.elapsed_time(b))
    return min(t)


def test_pair_search_of_a_cluster_is_not_serial(gpu):
    """10^5 droplets, uniform and in 1/20 of the box side, pairs that reach a tenth of their spacing."""
    import torch
    n = 100_000
    ms = {}
    for side in (1.0, 0.05):
        d, stb = _population(32, "f64", _rows(n, side))
        reach = 0.1 * side * 2 * np.pi / n ** (1 / 3)
        rad = torch.full((n,), 0.5 * reach, dtype=torch.float64, device=gpu)
        ms[side] = (_ms(lambda: stb.collision_pairs(rad)), _ms(lambda: stb.pair_statistics(reach, 8)))
        d.close()
    assert all(c < 25 * u for u, c in zip(ms[1.0], ms[0.05])), ms


@pytest.mark.parametrize("n,side", [(100, 0.02), (1500, 0.05), (3000, 0.3)])
def test_pairs_of_a_cluster_against_brute_force(gpu, n, side):
    """Short reaches: coarse cells, or those that the reach allows when the droplets crowd."""
    import torch
    from oracle import collide
    rows = _rows(n, side, n)
    d, stb = _population(32, "f64", rows)
    L = 2 * np.pi
    for near in (0.4, 0.05):
        r = near * side * L / n ** (1 / 3)
        rad = np.random.default_rng(n).uniform(0.5 * r, r, n)
        got = stb.collision_pairs(torch.from_numpy(rad).to(gpu)).cpu().numpy()
        want = collide.pairs_bruteforce(rows, rad, L)
        assert np.array_equal(got, want) and (near < 0.1 or len(want))
        assert np.array_equal(stb.pair_statistics(2 * r, 9)["counts"], collide.pair_stats_bruteforce(rows, L, 2 * r, 9)[0])
    d.close()


def test_captured_pair_statistics(gpu):
    """A call under capture cannot wait for the device: it replays what the eager call counts."""
    import torch
    from lucky_droplets_amd import _lib
    rows = _rows(2000, 0.1)
    d, stb = _population(32, "f64", rows)
    want = stb.pair_statistics(0.02, 16)["counts"]
    buf = torch.zeros((3, 16), dtype=torch.float64, device=gpu)

    def call():
        d._stream()
        _lib.check(d.lib.ld_pair_stats(d.ctx, stb.coord.data_ptr(), 2000, 0.02, 16, buf[0].data_ptr(),
                                       buf[1].data_ptr(), buf[2].data_ptr()))

    call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call()
    for _ in range(3):
        buf.fill_(7.0)
        g.replay()
        stb.pair_statistics(0.3, 16)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(buf[0].cpu().numpy().view(np.int64), want)
    d.close()
