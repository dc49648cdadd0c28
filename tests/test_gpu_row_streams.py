"""Row calls (interp, exterp, pRHS) that sort their rows share scratch memory of
the context with each other and with the steps: calls on several streams, and
calls captured into a graph, give what they give alone.

interp and RK4 are compared bit by bit (a row's sum does not depend on its
slot); deposits to 1e-12 of their largest value (FP64 sums in another order).
The two forms of the gather differ in the last bits, which shows the one taken."""
import numpy as np
import pytest

from helpers import inputs
from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu

N = 64


def _setup(gpu, npart, seed=0, sort_min=0, monkeypatch=None):
    import torch
    from lucky_droplets_amd.dns import ForcedDNS
    from lucky_droplets_amd.particles import MPI_particles
    monkeypatch.setenv("LD_ROW_SORT_MIN", str(sort_min))
    cfg = Config(N=N, precision="f64", nu=0.02, nshells=2, profile="k4", n_particles=npart,
                 st_dist=("uniform", 0.05, 1.0), gravity=True)
    uk, n, coord, _ = inputs(cfg, seed=seed, n_noise=0.2)
    d = ForcedDNS(cfg)
    stb = MPI_particles(None, cfg.L, cfg.N, npart, cfg.sts, 0.05, cfg.g, cfg.nu_eff, cfg.tf, cfg.rhop, cfg.M0, dns=d,
                        coord=coord)
    f = torch.randn((7, N, N, N), dtype=torch.float64, device=gpu, generator=torch.Generator(gpu).manual_seed(seed))
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(gpu)
    return d, stb, f, t(uk), t(n)


def _close(a, b):
    return float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


def test_captured_calls_keep_out_of_the_shared_scratch(gpu, monkeypatch):
    """A captured call takes the kernels without scratch, so a replay may run beside eager row
    calls and steps of the same context on another stream."""
    import torch
    npart = 30011
    d, stb, f, uk, n = _setup(gpu, npart, sort_min=1 << 40, monkeypatch=monkeypatch)
    plain = stb.interp_cosine(stb.coord, f).clone()
    d.close()
    d, stb, f, uk, n = _setup(gpu, npart, monkeypatch=monkeypatch)
    rows = stb.coord.clone()
    other = torch.roll(stb.coord, 1234, 0).contiguous()
    w = torch.rand((npart, 1), dtype=torch.float64, device=gpu, generator=torch.Generator(gpu).manual_seed(5))
    fc, fc2 = torch.empty_like(n), torch.empty_like(n)

    def calls():
        stb.exterpmat = w
        dep = stb.exterp_cosine_scalar(rows, fc)
        rhs = stb.pRHS(0.0, rows, f[:3], f[3:6], f[6], fc2, None)[1]
        return stb.interp_cosine(rows, f), dep, rhs

    eager = [x.clone() for x in calls()]
    assert not torch.equal(eager[0], plain)              # the eager call sorts
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = calls()
    side = torch.cuda.Stream()
    d.set_state(uk, n, rows)
    torch.cuda.synchronize()
    for it in range(6):
        for x in out:
            x.fill_(3.0)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):                    # eager users of the scratch beside the replay
            a = stb.interp_cosine(other, f)
        g.replay()
        with torch.cuda.stream(side):
            if it % 2:
                d.advance(1e-3, 1)
            b = stb.interp_cosine(other, f)
        torch.cuda.synchronize()
        assert torch.equal(out[0], plain)
        assert _close(out[1], eager[1]) and _close(out[2], eager[2])
        assert torch.equal(a, torch.roll(eager[0], 1234, 0)) and torch.equal(b, a)
    d.close()


def test_row_calls_on_several_streams(gpu, monkeypatch):
    """Sorted row calls alternate between streams, with RK4 and steps among them."""
    import torch
    npart = 50021
    d, stb, f, uk, n = _setup(gpu, npart, monkeypatch=monkeypatch)
    rows = [stb.coord.clone(), stb.coord.flip(0).contiguous(), torch.roll(stb.coord, 777, 0).contiguous()]
    stb.coord = rows[0]
    w = torch.rand((npart, 1), dtype=torch.float64, device=gpu, generator=torch.Generator(gpu).manual_seed(6))

    def row_calls(r):
        stb.exterpmat = w
        dep = stb.exterp_cosine_scalar(r, torch.empty_like(n))
        rhs, fc = stb.pRHS(0.0, r, f[:3], f[3:6], f[6], torch.empty_like(n), None)[1:]
        return stb.interp_cosine(r, f), rhs, dep, fc

    def rk4():
        return d.RK4(0.0, 0.01, stb, uk, n.clone())

    def steps():
        d.set_state(uk, n, rows[0])
        d.advance(1e-3, 2)
        out = (torch.empty_like(rows[0]), torch.empty_like(uk), torch.empty_like(n))
        d.get_state(out[1], out[2], out[0])
        return out

    jobs = [lambda r=r: row_calls(r) for r in rows] + [rk4, lambda: row_calls(rows[1]), steps, lambda: row_calls(rows[2]), rk4]
    state = (rk4, steps)                 # calls on the context's state: their own order is the caller's
    alone = []
    for j in jobs:
        alone.append([x.clone() for x in j()])
        torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    for turn in range(3):
        got, last = [], None
        for k, j in enumerate(jobs):
            with torch.cuda.stream(streams[(k + turn) % 3]):
                here = torch.cuda.current_stream()
                if j in state and last is not None:
                    here.wait_event(last)
                got.append(j())
                if j in state:
                    last = here.record_event()
        torch.cuda.synchronize()
        for k, (a, b) in enumerate(zip(got, alone)):
            exact = len(a) if len(a) == 3 else 2
            assert all(torch.equal(x, y) for x, y in zip(a[:exact], b[:exact])), (turn, k)
            assert all(_close(x, y) for x, y in zip(a[exact:], b[exact:])), (turn, k)
    d.close()
