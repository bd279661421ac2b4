"""Single-layer meshes whose y column transforms its even and odd ky one after the other (k_col of
csrc/fft_mixed.hip, in FP64 from 250 rows on): the lengths at both ends, 343 rows, whose 3 * 343 outputs are
five more than 128 lanes keep, and lengths around it, against the oracle: the FP64 path at 1e-12 of the
largest value, FP32 stencils (the same FP64 column, its field rounded to FP32) at 2e-7."""
import pytest

from test_gpu_parity import build, normwise, rand_m

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("f32_stencils", 2e-7)])
@pytest.mark.parametrize("n", [(5, 245, 1), (5, 250, 1), (5, 338, 1), (5, 343, 1), (40, 343, 1), (3, 350, 1), (2, 1365, 1),
                               (2, 1372, 1)], ids=lambda n: "x".join(map(str, n)))
def test_column_lengths(n, precision, tol):
    mesh = n + (2e-9, 2.5e-9, 3e-9)
    print(f"\n[column lengths] mesh={n} {precision}", flush=True)
    state, terms, sim = build(mesh, 1.1e6, rand_m(n, 61), [("demag", {})])
    h = terms[0].H_in_Apm(state, precision=precision)
    assert normwise(h, sim.heff()) <= tol, normwise(h, sim.heff())
