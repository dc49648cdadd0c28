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
