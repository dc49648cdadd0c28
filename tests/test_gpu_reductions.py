"""The diagnostics' reductions at the sizes where their splits end: shells of
white-noise fields (every mode of the half spectrum, corners included) and
statistics of columns that are not aligned for wide loads.  Sums of at most
3 N^2 (N/2 + 1) FP64 terms of one sign: relative rounding below 1e-12."""
import numpy as np
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


def _shells(N):
    k = np.fft.fftfreq(N, 1.0 / N)
    k2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + np.arange(N // 2 + 1)[None, None, :] ** 2
    w = np.full(N // 2 + 1, 2.0)
    w[0] = w[-1] = 1.0
    return k2, np.round(np.sqrt(k2)).astype(int), w * (2 * np.pi) ** 3 / float(N) ** 6


@pytest.mark.parametrize("N,prec,nf", [(16, "f64", 1), (16, "f32", 5), (32, "f32", 3), (64, "f64", 2), (128, "f32", 3)])
def test_shell_sums_of_white_noise(gpu, N, prec, nf):
    import torch
    from lucky_droplets_amd import _lib
    from lucky_droplets_amd.dns import ForcedDNS, _ptr
    d = ForcedDNS(Config(N=N, precision=prec, nu=0.02), max_particles=0)
    rng = np.random.default_rng(N + nf)
    f = rng.standard_normal((nf, N, N, N // 2 + 1)) + 1j * rng.standard_normal((nf, N, N, N // 2 + 1))
    fg = torch.from_numpy(f).to(gpu).to(d.cdtype).contiguous()
    f = fg.cpu().numpy().astype(np.complex128)
    k2, s, w = _shells(N)
    ok = s <= N // 2

    def bins(x, sel=ok):
        return np.bincount(s[sel], weights=x[sel], minlength=N // 2 + 1)

    p = (np.abs(f) ** 2).sum(0) * w
    got = d.spectrum(fg, 0.25).cpu().numpy()
    assert np.max(np.abs(got - bins(0.25 * p)) / bins(0.25 * p)) < 1e-12
    if nf >= 3:
        u = fg[:3].contiguous()
        q = (np.abs(f[:3]) ** 2).sum(0) * w
        got = d.dissipation(u).cpu().numpy()
        ref = bins(0.02 * k2 * q)
        assert np.max(np.abs(got - ref)) < 1e-12 * ref.max()
        out = torch.empty(N // 2 + 1, dtype=torch.float64, device=gpu)
        d._stream()
        _lib.check(d.lib.ld_flux(d.ctx, _ptr(u), _ptr(u), _ptr(out)))
        ref = np.cumsum(bins(q, ok & (s <= N / 3))[::-1])[::-1]
        assert np.max(np.abs(out.cpu().numpy() - ref)) < 1e-12 * ref.max()
    d.close()


@pytest.mark.parametrize("prec,npart", [("f32", 1), ("f32", 3), ("f64", 5), ("f32", 4099), ("f64", 20001)])
def test_statistics_of_unaligned_columns(gpu, prec, npart):
    """The mass column starts at 3 x capacity entries: with an odd capacity it is aligned to one entry only."""
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    cfg = Config(N=16, precision=prec, nu=0.02, n_particles=npart)
    d = ForcedDNS(cfg)
    rng = np.random.default_rng(npart)
    rows = rng.uniform(0.1, 1.0, (npart, 7))
    d.set_state(d.zeros_spec(3), d.zeros_real().fill_(1.0), torch.from_numpy(rows).to(gpu))
    m = rows[:, 6].astype(np.float32 if prec == "f32" else np.float64).astype(np.float64)
    got = d.droplet_stats()
    ref = (m.sum(), m.min(), m.max(), (m * m).sum())
    assert all(abs(a - b) <= 1e-12 * abs(b) for a, b in zip(got, ref))
    x = torch.from_numpy(rng.standard_normal((2, 16, 16, 16))).to(gpu).to(d.rdtype)
    xr = x.double().cpu().numpy()
    got = d.field_stats(x)
    assert got[1] == xr.min() and got[2] == xr.max() and abs(got[3] - (xr ** 2).sum()) < 1e-12 * (xr ** 2).sum()
    d.close()
