"""ld_pair_stats returns before the device is done, also where the number of
cells depends on how the droplets lie (as it does not under capture, where
nothing can be waited for)."""
import numpy as np
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


# fewer cells than the reach allows: droplets spread over the box, half of them in a corner, all of them
@pytest.mark.parametrize("inside", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("n", [2, 300, 4000])
def test_pair_statistics_do_not_wait(gpu, n, inside):
    import torch
    from oracle import collide
    from lucky_droplets_amd import _lib
    from lucky_droplets_amd.dns import ForcedDNS
    L, bins = 2 * np.pi, 7
    rng = np.random.default_rng(n)
    rows = rng.uniform(0, L, (n, 7))
    k = int(inside * n)
    rows[:k, :3] = rows[:k, :3] * 0.05 + 6.1                 # across the box's faces
    reach = 0.5 * (0.05 if k else 1.0) * L / n ** (1 / 3)
    d = ForcedDNS(Config(N=32, precision="f64", nu=0.02, n_particles=n))
    coord = torch.from_numpy(rows).to(gpu)
    counts = torch.zeros(bins, dtype=torch.int64, device=gpu)
    w = torch.zeros((2, bins), dtype=torch.float64, device=gpu)

    def call(r):
        d._stream()
        _lib.check(d.lib.ld_pair_stats(d.ctx, coord.data_ptr(), n, r, bins, counts.data_ptr(), w[0].data_ptr(),
                                       w[1].data_ptr()))

    call(reach)                                              # allocates the workspaces
    torch.cuda.synchronize()
    for r in (reach, 0.2 * reach, reach):
        r = max(r, 0.03)
        busy = torch.cuda.Event()
        torch.cuda._sleep(200_000_000)                       # about 0.1 s
        busy.record()
        call(r)
        assert not busy.query()
        torch.cuda.synchronize()
        assert np.array_equal(counts.cpu().numpy(), collide.pair_stats_bruteforce(rows, L, r, bins)[0])
    d.close()
