"""Demag fields of films whose y and z stages run as one column pass (csrc/fft_slab.hip): every row
count it takes, with one and several lines per wave, classes and partly filled last waves, against the
oracle.  Tolerances as for every field of these paths: FP64 1e-12 of the largest value, FP32 1e-5
against the FP64 field on the FP32 path's own tensor."""
import pytest

from test_gpu_parity import build, mf, normwise, rand_m

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [2, 3, 4, 8])
@pytest.mark.parametrize("ny", [64, 128, 256, 512, 1024])
def test_slab_field(ny, nz):
    check(({64: 9, 128: 20, 256: 6, 512: 3, 1024: 2}[ny], ny, nz))


@pytest.mark.parametrize("n", [(128, 64, 2), (150, 64, 3), (256, 64, 2), (300, 128, 2), (260, 1024, 2), (70, 1024, 3)],
                         ids=lambda n: "x".join(map(str, n)))
def test_slab_shared_columns(n):
    """Columns whose classes several work-groups share: all of them, the last round's, none."""
    check(n)


def check(n):
    mesh = n + (2e-9, 2.5e-9, 3e-9)
    print(f"\n[slab] mesh={n}", flush=True)
    state, terms, sim = build(mesh, 1.1e6, rand_m(n, 31), [("demag", {})])
    M = mf()
    h64 = terms[0].H_in_Apm(state)
    assert normwise(h64, sim.heff()) <= 1e-12
    oct64 = M.DemagField(terms[0].mesh, octant_tensor=True).H_in_Apm(state)
    assert normwise(terms[0].H_in_Apm(state, precision="f32"), oct64) <= 1e-5
