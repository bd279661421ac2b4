"""RKKY weights stored as indices into a table of the distinct sets of six weights, and in full where the
sets do not fit it: few materials, about as many sets as the table has places, and random couplings,
changed from one form to the other on a live context.  Against the oracle at the tolerances of the
stencils (FP64 1e-12, FP32 1e-5 of the largest value)."""
import numpy as np
import pytest

from test_gpu_parity import build, normwise, rand_m

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(7, 5, 3), (256, 3, 4)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("sets", [1, 40, 10 ** 9])
def test_rkky_sets(n, sets):
    rng = np.random.default_rng(5)
    mesh = n + (2e-9, 2.5e-9, 3e-9)
    print(f"\n[rkky sets] mesh={n} {sets}", flush=True)

    def materials(count):
        A = 1.3e-11 * (1 + rng.random(n)) if count > n[0] * n[1] * n[2] else \
            1.3e-11 * (1 + rng.integers(0, count, n) / count)
        return np.full(n, -1e-12), A

    rk, A = materials(sets)
    state, terms, sim = build(mesh, 1e6, rand_m(n, 41), [("rkky", {"rk": rk, "A": A})])
    for precision, tol in (("f64", 1e-12), ("f32", 1e-5)):
        assert normwise(terms[0].H_in_Apm(state, precision=precision), sim.heff()) <= tol
