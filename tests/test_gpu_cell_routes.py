"""Meshes of several layers take a lane per cell or walk z columns in the per-cell pass, by how many
work-groups they give (MAFX_NUM_CUS = 1 makes every mesh here walk columns): field and integrator steps of
both routes against the oracle, FP64 1e-12 and FP32 1e-5 of the largest field; steps of both routes against
each other, where each stage's field differs by rounding alone (1e-12 and 1e-7 of m after three steps of
1e-14 s, which turn m by some 1e-3)."""
import numpy as np
import pytest

from test_gpu_parity import build, mf, normwise, rand_m

pytestmark = pytest.mark.gpu

LISTS = {
    "chiral": [("demag", {}), ("exchange", {"A": 1.5e-11}), ("dmi", {"D": 3e-3}), ("uniaxial", {"K": 8e5})],
    "permalloy": [("demag", {}), ("exchange", {"A": 1.3e-11}), ("zeeman_h", {"h": (1e4, 2e3, 0.0)})],
    "film": [("demag", {}), ("exchange", {"A": 1.5e-11}), ("dmi", {"D": 2e-3}), ("uniaxial", {"K": 5e5}),
             ("zeeman_h", {"h": (0.0, 0.0, 1e5)})],
    "multilayer": [("demag", {}), ("rkky", None), ("dmi", {"D": 2.5e-3}), ("uniaxial", {"K": 7e5}),
                   ("zeeman_h", {"h": (4e4, 0.0, 0.0)})],
    "other": [("exchange", {"A": 1.3e-11}), ("uniaxial", {"K": 5e5}), ("dmi", {"D": 1e-3})],
}


@pytest.mark.parametrize("n", [(256, 3, 2), (512, 2, 3), (256, 5, 5)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("terms", sorted(LISTS))
@pytest.mark.parametrize("precision,tol,step_tol", [("f64", 1e-12, 1e-12), ("f32", 1e-5, 1e-7)])
def test_cell_routes(n, terms, precision, tol, step_tol, monkeypatch):
    mesh = n + (2e-9, 2e-9, 3e-9)
    print(f"\n[cell routes] mesh={n} {terms} {precision}", flush=True)
    M = mf()
    rkky = {"rk": np.full(n, -1e-12), "A": 1e-11 * (1 + np.random.default_rng(3).integers(0, 3, n))}
    specs = [(k, rkky if kw is None else kw) for k, kw in LISTS[terms]]
    ends = []
    for cus in (None, "1"):
        if cus:
            monkeypatch.setenv("MAFX_NUM_CUS", cus)
        state, tl, sim = build(mesh, 8e5, rand_m(n, 51), specs)
        llg = M.LLGIntegrator(0.1, tl, "DP45", hmin=1e-14, hmax=1e-14, precision=precision)
        assert normwise(llg.H_in_Apm(state), sim.heff()) <= tol
        for _ in range(3):
            llg.step(state)
        ends.append(np.array(state.m))
    assert np.max(np.abs(ends[0] - ends[1])) <= step_tol
