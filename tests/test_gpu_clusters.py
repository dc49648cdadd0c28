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


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("counts", [(0, 1, 1024, 1025, 3000, 2047, 5, 4096), (9000, 0, 0, 0, 0, 0, 0, 0), (1,) * 7 + (7000,)])
def test_tiles_of_more_rows_than_a_block_takes(gpu, prec, counts, monkeypatch):
    """Rows per tile around the 1024 that a tile's block takes, against the gather by four lanes per row (the same
    weights and 64 products in another order: 1e-12 of the largest value)."""
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    monkeypatch.setenv("LD_ROW_SORT_MIN", "0")
    N = 32
    rng = np.random.default_rng(sum(counts))
    h = np.pi                                            # a tile's side: 16 of the 32 cells
    rows = np.concatenate([np.concatenate([rng.uniform(0, h, (c, 3)) + h * np.array([t >> 2, t >> 1 & 1, t & 1]),
                                           rng.uniform(0.1, 1.0, (c, 4))], 1) for t, c in enumerate(counts)])
    rows = rows[rng.permutation(len(rows))]
    fields = torch.from_numpy(rng.standard_normal((7, N, N, N))).to(gpu)
    got = []
    for line in (0, 1 << 40):
        monkeypatch.setenv("LD_ROW_TILE_MIN", str(line))
        d, stb = _population(N, prec, rows)
        f = fields.to(d.rdtype)
        out = [stb.interp_cosine(stb.coord, f).clone(), stb.interp_cosine(stb.coord, f[:1]).clone()]
        out.append(stb.pRHS(0.0, stb.coord, f[:3], f[3:6], f[6], torch.empty_like(f[0]), None)[1])
        out.append(stb.interpmat)
        got.append([x.cpu().numpy() for x in out])
        d.close()
    for a, b in zip(*got):
        assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))


def test_gather_of_a_cluster_is_not_serial(gpu):
    """10^6 rows at 128^3, uniform and in 1/20 of the box side."""
    import torch
    n, ms = 1_000_000, {}
    for side in (1.0, 0.05):
        d, stb = _population(128, "f32", _rows(n, side))
        f = torch.randn((7, 128, 128, 128), device=gpu)
        ms[side] = _ms(lambda: stb.interp_cosine(stb.coord, f))
        d.close()
    assert ms[0.05] < 5 * ms[1.0], ms


def _cluster_rows(N, n, k, seed):
    """n rows, k of them within one brick (16 cells, at its corner), the others uniform; unwrapped."""
    rng = np.random.default_rng(seed)
    rows = rng.uniform(0, 2 * np.pi, (n, 7))
    dx = 2 * np.pi / N
    rows[:k, :3] = 16 * dx + rng.uniform(-1.5, 14.5, (k, 3)) * dx
    rows[:, :3] += 2 * np.pi * rng.integers(-1, 2, (n, 3))
    rows[:, 6] = rng.uniform(0.05, 1.0, n) * 1e-3
    return rows[rng.permutation(n)]


# 8192 candidates stay with a brick's block; 64 shares at most (more than 64 x 8192 candidates in the last case)
@pytest.mark.parametrize("N,n,k", [(32, 8192, 8192), (32, 8193, 8193), (64, 20000, 8000), (64, 20000, 8190),
                                   (64, 40001, 30000), (64, 500_000, 450_000), (128, 700_000, 700_000)])
def test_deposits_of_crowded_bricks(gpu, N, n, k, monkeypatch):
    """Against one thread per row: positive FP64 terms, at most 10^6 a node in another order (1e-10 of the largest
    value; FP32 fields: that sum rounded once).  A weight that is not finite reaches its own 64 nodes."""
    import torch
    rows = _cluster_rows(N, n, k, n + k)
    w = torch.from_numpy(np.random.default_rng(n).uniform(0.1, 1.0, (n, 1))).to(gpu)
    bad = w.clone()
    bad[n // 2] = float("nan")
    got = {}
    for prec, line in (("f64", 1 << 40), ("f64", 0), ("f32", 0)):
        monkeypatch.setenv("LD_ROW_SORT_MIN", str(line))
        d, stb = _population(N, prec, rows)
        c = d.zeros_real()
        stb.exterpmat = bad
        poison = torch.isnan(stb.exterp_cosine_scalar(stb.coord, torch.full_like(c, 3.0))).cpu().numpy()
        stb.exterpmat = w
        dep = stb.exterp_cosine_scalar(stb.coord, torch.full_like(c, 3.0)).double().cpu().numpy()
        got[prec, line] = poison, dep
        d.close()
    p0, want = got["f64", 1 << 40]
    top = np.max(want)
    assert p0.any()
    for key, rel in ((("f64", 0), 0.0), (("f32", 0), 2.0 ** -24)):
        p, dep = got[key]
        assert np.array_equal(p, p0)
        assert np.all(np.abs(dep - want) <= 1e-10 * top + rel * np.abs(want)), key


def test_steps_after_a_crowded_deposit(gpu, monkeypatch):
    """The shares' scratch field is the fallback deposit's: it is zero again when RK4 uses it."""
    import torch
    from helpers import inputs
    from lucky_droplets_amd.dns import ForcedDNS
    from lucky_droplets_amd.particles import MPI_particles
    monkeypatch.setenv("LD_ROW_SORT_MIN", "0")
    n = 60_000
    cfg = Config(N=64, precision="f64", nu=0.02, nshells=2, profile="k4", n_particles=n,
                 st_dist=("uniform", 0.05, 1.0), gravity=True)
    uk, nn, coord, _ = inputs(cfg, seed=3, n_noise=0.2)
    crowd = torch.from_numpy(_cluster_rows(64, n, n, 1)).to(gpu)
    rows = coord.copy()
    rows[:, 3:6] *= 60.0                                  # most leave their bins: fallback deposit
    out = []
    for first in (False, True):
        d = ForcedDNS(cfg)
        stb = MPI_particles(None, cfg.L, cfg.N, n, cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop, cfg.M0, dns=d,
                            coord=rows)
        if first:
            stb.exterpmat = torch.ones((n, 1), dtype=torch.float64, device=gpu)
            for _ in range(2):
                stb.exterp_cosine_scalar(crowd, d.zeros_real())
        t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(gpu)
        r, u1, n1 = d.RK4(0.0, 0.01, stb, t(uk), t(nn))
        out.append([x.cpu().numpy() for x in (r, u1, n1)])
        d.close()
    assert np.isfinite(out[0][2]).all()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


def test_deposit_of_a_cluster_is_not_serial(gpu):
    """10^6 rows at 128^3, uniform and in 1/20 of the box side."""
    import torch
    n, ms = 1_000_000, {}
    for side in (1.0, 0.05):
        d, stb = _population(128, "f32", _rows(n, side))
        c = d.zeros_real()
        stb.exterpmat = torch.rand((n, 1), dtype=torch.float64, device=gpu)
        ms[side] = _ms(lambda: stb.exterp_cosine_scalar(stb.coord, c))
        d.close()
    assert ms[0.05] < 15 * ms[1.0], ms
