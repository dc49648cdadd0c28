"""The sorted row path's scratch holds the context's capacity: more rows take the
kernels of one thread per row, whatever the rule for sorting says."""
import numpy as np
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


def test_rows_beyond_the_capacity_take_the_general_kernels(gpu, monkeypatch):
    """LD_ROW_SORT_MIN=0 sorts every call that fits: interp tells the two paths apart by its last
    bits (each exact for its path); deposits and growth agree to 1e-12 (FP64, sums in another order)."""
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    from lucky_droplets_amd.particles import MPI_particles
    N, npart = 32, 9000
    cfg = Config(N=N, precision="f64", nu=0.02, n_particles=4096)
    rng = np.random.default_rng(6)
    rows = rng.uniform(0, cfg.L, (npart, 7))
    rows[:, 6] = rng.uniform(0.05, 1.0, npart) ** 1.5 * cfg.factor
    f = torch.from_numpy(rng.standard_normal((7, N, N, N))).to(gpu)
    w = torch.from_numpy(rng.standard_normal((npart, 1))).to(gpu)
    got = {}
    for cap, line in ((4096, 0), (npart - 1, 0), (npart, 0), (npart, 1 << 40)):
        monkeypatch.setenv("LD_ROW_SORT_MIN", str(line))
        d = ForcedDNS(cfg, max_particles=cap)
        stb = MPI_particles(None, cfg.L, cfg.N, npart, cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop, cfg.M0,
                            dns=d, coord=rows)
        out = [stb.interp_cosine(stb.coord, f).clone()]
        stb.exterpmat = w
        out.append(stb.exterp_cosine_scalar(stb.coord, torch.empty_like(f[0])))
        _, rhs, fc = stb.pRHS(0.0, stb.coord, f[:3], f[3:6], f[6], torch.empty_like(f[0]), None)
        out += [rhs, stb.interpmat, fc]
        torch.cuda.synchronize()
        got[cap, line] = [x.cpu().numpy() for x in out]
        d.close()
    general = got[npart, 1 << 40]
    assert not np.array_equal(got[npart, 0][0], general[0])          # fits: sorted
    for cap in (4096, npart - 1):
        assert np.array_equal(got[cap, 0][0], general[0])
        assert np.array_equal(got[cap, 0][2], general[2]) and np.array_equal(got[cap, 0][3], general[3])
    for k in ((4096, 0), (npart - 1, 0), (npart, 0)):
        for a, b in zip(got[k], general):
            assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))
