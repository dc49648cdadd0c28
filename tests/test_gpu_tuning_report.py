"""The reported launch geometry is what runs."""
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,prec,slabs,lines", [(128, "f32", 1, 16), (256, "f32", 1, 32), (256, "f32", 16, 16),
                                                (256, "f64", 1, 8)])
def test_inverse_y_lines_without_autotuner(gpu, N, prec, slabs, lines, monkeypatch):
    """The inverse y passes take 32 lines per block from 256^3 FP32 (16 where a slab does not hold whole groups)."""
    from lucky_droplets_amd.dns import ForcedDNS
    monkeypatch.setenv("LD_SLABS", str(slabs))
    d = ForcedDNS(Config(N=N, precision=prec, nu=0.02, n_particles=0))
    assert d.tuning()[0] == lines and d.tuning_all()[0]["y_lines"] == lines
    d.close()
