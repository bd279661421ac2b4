"""Demag fields on meshes whose extents reach every radix, schedule length and tile choice of
csrc/fft_mixed.hip (the x and y passes, the single-layer y column in both its forms and in the
power-of-two one, the thick-mesh z column), and lines too long for them, against the oracle.
Tolerances as for every field of these paths: FP64 1e-12 of the largest value against the oracle, FP32
1e-5 against the FP64 field on the FP32 path's own tensor (its difference from the oracle's tensor is
the far-field rounding noise of both, 5e-5 on a row of 3000 cells in FP64 arithmetic as well)."""
import numpy as np
import pytest

from test_gpu_parity import build, mf, normwise, rand_m

pytestmark = pytest.mark.gpu

MESHES = [(15, 13, 1), (99, 22, 1), (210, 1, 3), (77, 9, 2), (144, 5, 1),           # x lengths
          (7, 900, 2), (3, 390, 4), (2, 1001, 1), (60, 700, 1), (4, 1100, 1),        # y lengths, split column
          (5, 128, 1), (9, 256, 1), (4, 512, 1), (3, 1024, 1), (600, 128, 1),        # power-of-two column
          (36, 45, 9), (2, 3, 40), (26, 14, 11), (1, 2, 300), (33, 8, 16),           # z column
          (3000, 2, 1)]                                                              # in-place x in FP64


@pytest.mark.parametrize("n", MESHES, ids=lambda n: "x".join(map(str, n)))
def test_demag_lengths(n):
    mesh = n + (2e-9, 2.5e-9, 3e-9)
    print(f"\n[demag lengths] mesh={n}", flush=True)
    state, terms, sim = build(mesh, 1.1e6, rand_m(n, 21), [("demag", {})])
    M = mf()
    ref = sim.heff()
    h64 = terms[0].H_in_Apm(state)
    assert normwise(h64, ref) <= 1e-12, normwise(h64, ref)
    h32 = terms[0].H_in_Apm(state, precision="f32")
    oct64 = M.DemagField(terms[0].mesh, octant_tensor=True).H_in_Apm(state)
    assert normwise(h32, oct64) <= 1e-5, normwise(h32, oct64)
    hfull = M.DemagField(terms[0].mesh, full_tensor=True).H_in_Apm(state, precision="f32")
    assert normwise(hfull, ref) <= 1e-5, normwise(hfull, ref)


@pytest.mark.parametrize("n", [(20, 15, 1), (64, 128, 1), (16, 512, 1), (12, 10, 10)], ids=lambda n: "x".join(map(str, n)))
def test_atomistic_dipole_lengths(n):
    mesh = n + (0.27e-9,) * 3
    print(f"\n[dipole lengths] mesh={n}", flush=True)
    state, terms, sim = build(mesh, 2.4e-23, rand_m(n, 22), [("atom_dipole", {})])
    assert normwise(terms[0].H_in_Apm(state), sim.heff()) <= 1e-12
