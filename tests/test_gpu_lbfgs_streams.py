"""No LBFGS run ends while work on its vectors may still be queued, on either context's stream: they stay with
the context for its next run."""
import ctypes as C

import pytest

from test_gpu_parity import mf, rand_m

pytestmark = pytest.mark.gpu


def test_failing_run_leaves_both_streams_idle():
    """A stalled run that has moved to its finish context ends with an error there: whatever that context's
    stream still holds is waited for, as the work space is handed back."""
    print("\n[lbfgs streams]", flush=True)
    import torch
    M = mf()
    from magnumaf import _abi
    n = (32, 16, 1)
    g = M.Mesh(*n, 2e-9, 2e-9, 2e-9)
    state = M.State(g, 8e5, rand_m(n, 52))
    side = torch.cuda.Stream()
    load = torch.ones(1 << 26, device="cuda")
    calls = {"first": 0, "finish": 0}

    def rising(s):
        # a field against m that grows with every evaluation: no torque, and no iteration lowers the energy
        calls["first"] += 1
        return -1e6 * calls["first"] * s.m

    def failing(s):
        calls["finish"] += 1
        if calls["finish"] < 3:
            return 0.0, 0.0, 0.0
        with torch.cuda.stream(side):
            for _ in range(2000):
                load.mul_(1.0)
        raise RuntimeError("planned")

    stalling = [M.ExchangeField(1.3e-11), M.ExternalField(rising)]
    failing_terms = [M.ExchangeField(1.3e-11), M.ExternalField(failing, homogeneous_callback=True)]
    ctx = M.Context(g, 8e5, None, stalling, "f32")
    with torch.cuda.stream(side):
        finish = M.Context(g, 8e5, None, failing_terms, "f64")
    torch.cuda.synchronize()
    L = _abi.lib()
    assert L.mafx_lbfgs_set_finish_context(ctx.h, finish.h) == 0
    E, st = C.c_double(), _abi.LbfgsStats()
    rc = L.mafx_lbfgs_minimize(ctx.h, C.c_void_p(state.m_dev.data_ptr()), 1e-20, 200, 0, 1e-12, C.byref(E), C.byref(st))
    idle = side.query()
    torch.cuda.synchronize()
    assert rc != 0 and calls["finish"] == 3, (rc, calls)
    assert idle
