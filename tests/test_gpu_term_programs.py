"""Energy sums and LBFGS runs on the compile-time term programs of csrc/field.hip (both per-cell
mappings: rows of whole work-groups and any other mesh) against the oracle, and against the same terms
in an order that has no program, whose fields differ by the order of the term sum alone."""
import numpy as np
import pytest

from test_gpu_parity import build, energy_scale, mf, rand_m

pytestmark = pytest.mark.gpu

H0 = 2e4
MICRO = [("demag", {}), ("exchange", {"A": 1.3e-11}), ("dmi", {"D": 2e-3}), ("uniaxial", {"K": 4e5}),
         ("zeeman_h", {"h": (0.0, H0, 2 * H0)})]
J = 1.6e-21
ATOMS = [("atom_exchange", {"J": J}), ("atom_uniaxial", {"K": 0.02 * J}), ("atom_dmi", {"D": 0.2 * J}),
         ("atom_dipole", {}), ("atom_zeeman_h", {"h": (0.0, 0.0, 8e5)})]


def specs_of(which, n):
    if which == "atoms":
        return ATOMS
    if which == "rkky":
        return [MICRO[0], ("rkky", {"rk": np.full(n, -1e-12), "A": np.full(n, 1.3e-11)})] + MICRO[2:]
    return {"film": MICRO, "film0": MICRO[:4], "sp4": [MICRO[0], MICRO[1], MICRO[4]]}[which]


@pytest.mark.parametrize("n", [(256, 5, 2), (300, 3, 1), (20, 15, 3)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("which", ["film", "film0", "sp4", "rkky", "atoms"])
def test_energies(which, n):
    print(f"\n[term programs] {which} {n}", flush=True)
    mesh = n + ((0.27e-9,) * 3 if which == "atoms" else (3e-9, 3e-9, 2e-9))
    Ms = 2.4e-23 if which == "atoms" else 8e5
    state, terms, sim = build(mesh, Ms, rand_m(n, 31), specs_of(which, n))
    E, parts = state._context(terms, "f64").energy(state.m_dev)
    E_ref, parts_ref = sim.energy()
    scale = np.max(np.abs(parts_ref)) if which == "atoms" else energy_scale(mesh, Ms, parts_ref)
    assert np.max(np.abs(parts - parts_ref)) <= 1e-12 * scale
    assert abs(E - E_ref) <= 1e-12 * scale


@pytest.mark.parametrize("n", [(256, 4, 1), (24, 10, 1)], ids=lambda n: "x".join(map(str, n)))
def test_minimize_program_and_loop(n):
    """Four LBFGS iterations of the film list on its program and, with the last two terms exchanged,
    on the run-time loop.  A film's iterates keep a last-bit difference of the field below 1e-13."""
    print(f"\n[term programs minimize] {n}", flush=True)
    M = mf()
    mesh, m, out = n + (3e-9, 3e-9, 2e-9), rand_m(n, 32), []
    for specs in (MICRO, MICRO[:3] + [MICRO[4], MICRO[3]]):
        state, terms, _ = build(mesh, 8e5, m, specs)
        M.LBFGS_Minimizer(terms, tol=1e-20, maxiter=4).minimize(state)
        out.append(state.m)
    assert np.max(np.abs(out[0] - out[1])) <= 1e-11
