"""Weight gradients of batches with more pixel tiles than the layers of 16 channel blocks have chunks by
default (csrc/net_shapes.hpp), against oracle/warmstart_net.py at the tolerances of the other shapes."""
import numpy as np
import pytest

import oracle_import  # noqa: F401
import warmstart_net as NR
from test_gpu_warmstart import _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(13, 8, 264), (33, 32, 40), (70, 16, 64)])
def test_gradients_of_large_batches(shape):
    print(f"\n[net batches] B,H,W={shape}", flush=True)
    net, used, x, t, xd, td = _setup(*shape, seed=14)
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
