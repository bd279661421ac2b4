"""RKKY arrays replaced on a live context: the weights go from indices into the table of distinct sets to
the full form and back, with about as many sets as the table has places in between.  Each field against
the oracle at the tolerances of the stencils (FP64 1e-12, FP32 1e-5 of the largest value), and the
context's device bytes follow the form that the term holds."""
import numpy as np
import pytest

from test_gpu_parity import build, mf, normwise, rand_m

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol,weight", [("f64", 1e-12, 8), ("f32", 1e-5, 4)])
@pytest.mark.parametrize("n", [(20, 15, 3), (256, 3, 4)], ids=lambda n: "x".join(map(str, n)))
def test_forms_change_on_a_live_context(n, precision, tol, weight):
    print(f"\n[rkky update] mesh={n} {precision}", flush=True)
    M = mf()
    rng = np.random.default_rng(17)
    N = n[0] * n[1] * n[2]
    mesh = n + (2e-9, 2.5e-9, 3e-9)
    g, m = M.Mesh(*mesh), rand_m(n, 43)
    rk = np.full(n, -1e-12)
    few, many = np.full(n, 1.3e-11), 1.3e-11 * (1 + rng.random(n))
    state, terms, sim = build(mesh, 1e6, m, [("rkky", {"rk": rk, "A": few})])
    ctx = state._context(terms, precision)
    nbytes = []
    for A in (few, many, few, many):
        terms[0].A = M._scalar_flat(A, g)
        ctx.refresh(state)
        _, _, sim = build(mesh, 1e6, m, [("rkky", {"rk": rk, "A": A})])
        h = ctx.heff(state.m_dev).cpu().numpy()
        assert normwise(h, sim.heff_flat()) <= tol, normwise(h, sim.heff_flat())
        nbytes.append(ctx.device_bytes())
    assert state._context(terms, precision) is ctx
    assert nbytes[0] == nbytes[2] and nbytes[1] == nbytes[3]
    # six weights per cell against one byte per cell and the table of 256 sets of eight
    assert nbytes[1] - nbytes[0] == 6 * N * weight - (N + 256 * 8 * weight)


@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("f32", 1e-5)])
@pytest.mark.parametrize("cells", [180, 255, 256, 257, 300])
def test_sets_near_the_table_size(cells, precision, tol):
    """Every cell of a row has a set of its own: as many sets as cells."""
    print(f"\n[rkky table] cells={cells} {precision}", flush=True)
    n = (cells, 1, 1)
    rng = np.random.default_rng(cells)
    specs = [("rkky", {"rk": np.full(n, -1e-12), "A": 1.3e-11 * (1 + rng.random(n))})]
    state, terms, sim = build(n + (2e-9, 2.5e-9, 3e-9), 1e6, rand_m(n, 44), specs)
    h = terms[0].H_in_Apm(state, precision=precision)
    assert normwise(h, sim.heff()) <= tol, normwise(h, sim.heff())
