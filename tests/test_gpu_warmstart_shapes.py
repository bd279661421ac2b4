"""The matrix-core convolutions of csrc/net.hip at the edges of their tiles: image sides that are no
multiple of the 16- or 8-pixel tiles at any level, levels down to one cell, batches, and sizes large
enough for the unsplit form at every layer, against oracle/warmstart_net.py at the BF16 weights.
Tolerances: exact products in FP32 sums of up to 9 * 256 terms over eight layers, 8 * sqrt(2304) *
2^-24 = 2.3e-5 of the largest partial sums, times about 10 for their size over the result."""
import numpy as np
import pytest

import oracle_import  # noqa: F401
import warmstart_net as NR
from test_gpu_warmstart import _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 8, 8), (2, 40, 72), (3, 48, 24), (1, 8, 264), (8, 192, 184)])
def test_forward_at_tile_edges(shape):
    print(f"\n[net forward] B,H,W={shape}", flush=True)
    net, used, x, t, xd, td = _setup(*shape, seed=11)
    m = net.forward(xd).cpu().numpy()
    ref, _ = NR.forward(used, x.astype(np.float64))
    assert np.max(np.abs(m - ref)) <= 2e-4, np.max(np.abs(m - ref))


@pytest.mark.parametrize("shape", [(1, 8, 8), (2, 40, 72), (9, 48, 24), (1, 8, 136)])
def test_gradients_at_tile_edges(shape):
    print(f"\n[net gradients] B,H,W={shape}", flush=True)
    net, used, x, t, xd, td = _setup(*shape, seed=12)
    loss, g = net.gradients(xd, td)
    ref_loss, ref_grads, _ = NR.loss_and_grads(used, x.astype(np.float64), t.astype(np.float64))
    assert abs(loss - ref_loss) <= 1e-5 * abs(ref_loss)
    off = 0
    for layer, (dw, db) in enumerate(ref_grads):
        for ref in (dw, db):
            got = g[off:off + ref.size].reshape(ref.shape)
            off += ref.size
            err = np.linalg.norm(got - ref) / max(np.linalg.norm(ref), 1e-30)
            assert err <= 1e-3, (layer, ref.shape, err)
    assert off == g.size


def test_infinite_input_stays_infinite():
    """An infinite activation is not split into infinity - infinity: the cells it does not reach are
    unchanged."""
    import torch
    net, used, x, t, xd, td = _setup(1, 64, 64, seed=13)
    clean = net.forward(xd).cpu().numpy()
    xd[0, 0, 0, 0] = float("inf")
    m = net.forward(xd).cpu().numpy()
    torch.cuda.synchronize()
    # the receptive field of the four levels and back spans fewer than 48 cells
    assert np.array_equal(m[:, :, 56:, 56:], clean[:, :, 56:, 56:])
