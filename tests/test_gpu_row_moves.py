"""Fields to rows and subgrid rows: vector and scalar forms (row lengths that
are and are not multiples of four, row pointers off a 16-byte boundary) and the
ratios, against numpy.  The values are moved or take one FP32 multiply-add:
2^-23 of the operands."""
import ctypes

import numpy as np
import pytest

from lucky_droplets_amd.config import Config

pytestmark = pytest.mark.gpu


def _ctx(N, prec):
    from lucky_droplets_amd.dns import ForcedDNS
    return ForcedDNS(Config(N=N, precision=prec, nu=0.02), max_particles=0)


def _p(t, off=0):
    return ctypes.c_void_p(t.data_ptr() + off)


@pytest.mark.parametrize("N,prec,nc,off", [(16, "f32", 1, 0), (16, "f64", 3, 0), (32, "f32", 12, 0), (32, "f32", 12, 4),
                                           (16, "f64", 32, 0), (64, "f32", 6, 8)])
def test_fields_to_rows(gpu, N, prec, nc, off):
    import torch
    d = _ctx(N, prec)
    f = torch.randn((nc, N, N, N), device=gpu, dtype=d.rdtype)
    buf = torch.full((N ** 3 * nc + 8,), np.nan, dtype=torch.float32, device=gpu)
    d._stream()
    assert d.lib.ld_fields_to_rows(d.ctx, _p(f), nc, _p(buf, off), 0.5) == 0
    b = buf.cpu().numpy()
    k = off // 4
    ref = (f.cpu().numpy().reshape(nc, -1).T.astype(np.float32) * np.float32(0.5)).ravel()
    assert np.array_equal(b[k:k + ref.size], ref)
    assert np.isnan(b[:k]).all() and np.isnan(b[k + ref.size:]).all()
    d.close()


@pytest.mark.parametrize("N,prec,r,off", [(16, "f32", 1, 0), (16, "f32", 2, 0), (32, "f64", 2, 0), (32, "f32", 2, 4),
                                          (16, "f32", 4, 0), (64, "f32", 2, 0)])
def test_subgrid_rows(gpu, N, prec, r, off):
    import torch
    d = _ctx(N, prec)
    Nc, r3 = N // r, r ** 3
    fine = torch.randn((3, N, N, N), device=gpu, dtype=d.rdtype)
    base = torch.randn((3, N, N, N), device=gpu, dtype=d.rdtype)
    buf = torch.full((Nc ** 3 * 3 * r3 + 8,), np.nan, dtype=torch.float32, device=gpu)
    k, n = off // 4, Nc ** 3 * 3 * r3
    d._stream()
    assert d.lib.ld_subgrid_residual(d.ctx, _p(fine), _p(base), r, _p(buf, off), 2.0) == 0
    b = buf.cpu().numpy()
    res = (fine - base).float().mul(2.0).cpu().numpy()
    rows = res.reshape(3, Nc, r, Nc, r, Nc, r).transpose(1, 3, 5, 0, 2, 4, 6).reshape(-1)
    assert np.array_equal(b[k:k + n], rows)
    assert np.isnan(b[:k]).all() and np.isnan(b[k + n:]).all()
    out = torch.empty_like(base)
    assert d.lib.ld_subgrid_compose(d.ctx, _p(buf, off), r, _p(base), _p(out), 0.5) == 0
    ref = base.double().cpu().numpy() + 0.5 * res.astype(np.float64)
    assert np.max(np.abs(out.double().cpu().numpy() - ref)) <= 2.0 ** -23 * np.max(np.abs(ref))
    d.close()
