"""The LBFGS work space that a context keeps between runs: counted in its device bytes up to the bound of
256 MiB, not held beyond it."""
import pytest

from test_gpu_parity import mf, rand_m

pytestmark = pytest.mark.gpu


def vectors(n):
    """7 + 2 (5 + 1) vectors of 3N doubles in whole 256-byte lines, and 16 scalars."""
    return 19 * ((24 * n + 255) // 256 * 256) + 128


@pytest.mark.parametrize("n,kept", [((16, 12, 1), True), ((61, 33, 2), True), ((800, 800, 1), False)],
                         ids=lambda v: str(v))
def test_kept_workspace_is_counted(n, kept):
    print(f"\n[lbfgs workspace] mesh={n}", flush=True)
    M = mf()
    state = M.State(M.Mesh(*n, 2e-9, 2e-9, 2e-9), 8e5, rand_m(n, 51))
    terms = [M.ExchangeField(1.3e-11), M.UniaxialAnisotropyField(5e5, [0, 0, 1])]
    ctx = state._context(terms, "f64")
    before = ctx.device_bytes()
    for _ in range(2):
        M.LBFGS_Minimizer(terms, tol=1e-20, maxiter=2).minimize(state)
        assert state._context(terms, "f64") is ctx
        assert ctx.device_bytes() - before == (vectors(n[0] * n[1] * n[2]) if kept else 0)
