"""The column pass of csrc/fft_slab.hip at every row count, layer count and precision it has a kernel for,
on meshes that take it whatever the rules on full launches say: MAFX_NUM_CUS sets the CU count those rules
see.  With one CU every mesh has whole rounds of columns; with two CUs and 3 columns (and three CUs and 5)
the one (two) columns of the last round are shared by classes.  Each run asserts that the pass was launched,
by its profile entry.  And the separate y passes of the meshes without one, whose persistent forward pass
takes many tiles per group with one CU.

Tolerances as for every field of these paths: FP64 1e-12 of the largest value against the oracle, FP32 1e-5
against the FP64 field on the FP32 path's own tensor."""
import numpy as np
import pytest

from test_gpu_parity import build, mf, normwise, rand_m

pytestmark = pytest.mark.gpu

# every (rows, layers) with a kernel: FP32 without 1024 x 8, FP64 without 8 layers of 256 rows or more
KERNELS = [(ny, nz, p) for p in ("f32", "f64") for ny in (64, 128, 256, 512, 1024) for nz in (2, 3, 4, 8)
           if nz < 8 or ny < (1024 if p == "f32" else 256)]


def field_twice(state, term, precision):
    """The field of two evaluations of one context, equal to the last bit, and the kernels they ran."""
    ctx = state._context([term], precision)
    ctx.prof_reset()
    ctx.prof(True)
    h = [ctx.heff(state.m_dev).cpu().numpy() for _ in range(2)]
    rows = ctx.prof_report()
    ctx.prof(False)
    assert np.array_equal(h[0].view(np.uint64), h[1].view(np.uint64))
    return h[0], rows


def check(n, precision):
    M = mf()
    mesh = n + (2e-9, 2.5e-9, 3e-9)
    state, terms, sim = build(mesh, 1.1e6, rand_m(n, 33), [("demag", {})])
    if precision == "f64":
        h, rows = field_twice(state, terms[0], "f64")
        ref, tol = sim.heff_flat(), 1e-12
    else:
        h, rows = field_twice(state, terms[0], "f32")
        ref, tol = state._context([M.DemagField(M.Mesh(*mesh), octant_tensor=True)], "f64").heff(state.m_dev).cpu().numpy(), 1e-5
    assert normwise(h, ref) <= tol, normwise(h, ref)
    return rows


@pytest.mark.parametrize("ny,nz,precision", KERNELS)
def test_every_column_kernel(ny, nz, precision, monkeypatch):
    n = (2, ny, nz)
    print(f"\n[column pass] mesh={n} {precision}", flush=True)
    monkeypatch.setenv("MAFX_NUM_CUS", "1")
    rows = check(n, precision)
    assert f"slab_{precision}" in rows and not any(r.startswith("fft_y") for r in rows), sorted(rows)


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n,cus", [((2, 1024, 2), 2), ((4, 1024, 3), 3), ((2, 1024, 4), 2), ((4, 512, 4), 3),
                                   ((4, 64, 8), 3)], ids=str)
def test_shared_columns(n, cus, precision, monkeypatch):
    print(f"\n[shared columns] mesh={n} cus={cus} {precision}", flush=True)
    monkeypatch.setenv("MAFX_NUM_CUS", str(cus))
    rows = check(n, precision)
    assert f"slab_{precision}" in rows, sorted(rows)


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_shared_columns_on_a_side_stream(precision, monkeypatch):
    """A context created and used at once on a stream of its own, which does not wait for the null stream."""
    import torch
    print(f"\n[shared columns, side stream] {precision}", flush=True)
    monkeypatch.setenv("MAFX_NUM_CUS", "3")
    M = mf()
    n = (4, 512, 4)
    g = M.Mesh(*n, 2e-9, 2.5e-9, 3e-9)
    state = M.State(g, 1.1e6, rand_m(n, 35))
    term = M.DemagField(g)
    ref = state._context([term], precision).heff(state.m_dev).cpu().numpy()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        ctx = M.Context(g, 1.1e6, None, [term], precision)
        h = ctx.heff(state.m_dev)
        side.synchronize()
        assert np.array_equal(h.cpu().numpy().view(np.uint64), ref.view(np.uint64))


@pytest.mark.parametrize("n,precision,column", [((27, 1024, 2), "f32", False), ((30, 1024, 2), "f32", True),
                                                ((25, 256, 3), "f64", False), ((22, 256, 3), "f64", True),
                                                ((64, 256, 3), "f64", True), ((25, 256, 3), "f32", True)], ids=str)
def test_rounds_of_columns(n, precision, column, monkeypatch):
    """With eight CUs: the two shapes that gain least leave the pass to well filled, or few, rounds."""
    print(f"\n[rounds] mesh={n} {precision}", flush=True)
    monkeypatch.setenv("MAFX_NUM_CUS", "8")
    rows = check(n, precision)
    assert (f"slab_{precision}" in rows) == column, sorted(rows)


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n", [(256, 256, 5), (64, 1024, 5), (32, 1024, 8), (16, 512, 12)], ids=lambda n: "x".join(map(str, n)))
def test_separate_y_passes_bitwise(n, precision, monkeypatch):
    """One resident set of groups, each taking many tiles, against one tile per group, bit for bit."""
    print(f"\n[y passes] mesh={n} {precision}", flush=True)
    M = mf()
    g = M.Mesh(*n, 2e-9, 1e-9, 2e-9)
    m = rand_m(n, 34)
    ends = []
    for cus in (None, "1"):
        if cus:
            monkeypatch.setenv("MAFX_NUM_CUS", cus)
        state = M.State(g, 1.1e6, m)
        h, rows = field_twice(state, M.DemagField(g, device_tensor=True), precision)
        assert f"fft_y_fwd_{precision}" in rows and f"fft_y_inv_{precision}" in rows, sorted(rows)
        ends.append(h)
    assert np.array_equal(ends[0].view(np.uint64), ends[1].view(np.uint64))
