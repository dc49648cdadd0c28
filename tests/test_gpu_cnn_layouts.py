"""The CNN's activation layouts: every grid size class (N < 16 channels-last;
16, 32 and >= 64 with 1, 2 and 4 node tiles per segment; 128 with two segments
per z-line) and channel counts that pad, fill and split the 16- and 32-channel
tiles, output rows aligned and not.  One layer, so no rounding to bfloat16
after the FP32 sums: 27 x 32 products of unit variance in another order differ
by less than 864 x 2^-24 < 6e-5 of the largest value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,ci,co", [(4, 3, 5), (8, 32, 32), (16, 1, 4), (16, 17, 3), (32, 5, 24), (32, 32, 1),
                                     (64, 12, 17), (64, 16, 16), (64, 32, 32), (128, 20, 8)])
def test_single_layer_rows(gpu, N, ci, co):
    import ctypes
    import torch
    from lucky_droplets_amd import _lib
    from lucky_droplets_amd.cnn import SubgridCNN
    from oracle import cnn as ocnn
    rng = np.random.default_rng(N + ci + co)
    layers = [(rng.standard_normal((27, co, ci)).astype(np.float32), rng.standard_normal(co).astype(np.float32))]
    x = rng.standard_normal((N, N, N, ci)).astype(np.float32)
    net = SubgridCNN(N, (ci, co))
    net.set_params(layers)
    xg = torch.from_numpy(x).to(gpu)
    y = net.forward(xg).cpu().numpy()
    # rows starting 4 bytes after a 16-byte boundary
    buf = torch.full((N ** 3 * co + 2,), np.nan, dtype=torch.float32, device=gpu)
    net._stream()
    _lib.check(net.lib.ld_cnn_forward(net.h, ctypes.c_void_p(xg.data_ptr()), ctypes.c_void_p(buf.data_ptr() + 4)))
    b = buf.cpu().numpy()
    assert np.isnan(b[0]) and np.isnan(b[-1]) and np.array_equal(b[1:-1], y.ravel())
    if N <= 32:
        nodes = np.stack(np.meshgrid(*[np.arange(N)] * 3, indexing="ij"), -1).reshape(-1, 3)
    else:
        nodes = np.concatenate([rng.integers(0, N, (400, 3)),
                                [[a, b_, c] for a in (0, N - 1) for b_ in (0, N - 1) for c in (0, 1, 63, N - 2, N - 1)]])
    ref = ocnn.forward_at(layers, x, nodes, bf16=True)
    got = y.reshape(N, N, N, co)[nodes[:, 0], nodes[:, 1], nodes[:, 2]]
    assert np.max(np.abs(got - ref)) < 6e-5 * np.max(np.abs(ref))
    net.close()


@pytest.mark.parametrize("N,ch", [(8, (2, 16, 3)), (16, (5, 32, 16, 4)), (32, (17, 16, 32, 1)), (64, (3, 32, 32, 24))])
def test_gradients_match_oracle(gpu, N, ch):
    """Tolerances of the network's parity test: bfloat16 rounding ties of activations and back-propagated gradients."""
    import torch
    from lucky_droplets_amd.cnn import SubgridCNN
    from oracle import cnn as ocnn
    rng = np.random.default_rng(N)
    layers = [(rng.normal(0, np.sqrt(2.0 / (27 * a)), (27, b, a)).astype(np.float32),
               rng.normal(0, 0.1, b).astype(np.float32)) for a, b in zip(ch[:-1], ch[1:])]
    x = rng.standard_normal((N, N, N, ch[0])).astype(np.float32)
    t = rng.standard_normal((N, N, N, ch[-1])).astype(np.float32)
    net = SubgridCNN(N, ch)
    net.set_params(layers)
    loss, g = net.grad(torch.from_numpy(x).to(gpu), torch.from_numpy(t).to(gpu))
    lr, gr = ocnn.loss_and_grads(layers, x, t, bf16=True)
    assert abs(loss - lr) < 1e-2 * lr
    for (gw, gb), (rw, rb) in zip(net.unpack(g.cpu().numpy()), gr):
        assert np.linalg.norm(gw - rw) / np.linalg.norm(rw) < 3e-2
        assert np.linalg.norm(gb - rb) / max(np.linalg.norm(rb), 1e-30) < 3e-2
    net.close()
