"""The FP64 grid stage on product grids (csrc/separable.hpp): densities and
dH_sp of the factorised contractions against the oracle, whose sums run over
all grid points at once.

The sizes cross every edge of the kernels: axial points below, at and above a
16-column tile of (re, im) pairs, a 64-lane wave and the five tiles of a column
group; radial points that are no multiple of the 4-point step or the 16-row
tile; blocks with one radial function and with several.  The bar is that of the
other FP64 units, 1e-12 of each array's largest element: both sides sum a few
thousand FP64 terms, some 1e-15 each.  A basis whose tables are no products
must take the general kernels and give their results."""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ARG = [0, 1, 2, 3, 6, 7, 4, 5]   # quadrant slots <-> calc_dHsp_interface argument order
COUPLINGS = dict(vpair_t0=-346.352, override_cs0=128.279, override_csr=0.0, override_cds=0.0)


def problem(nsh, ngh, ngl, op="GT", K=0, Z=20, N=28, beta=0.0, beta_type="-", **kw):
    from pynfam_amd.problem import build_problem
    from pynfam_amd.synthetic import synthetic_basis
    basis = synthetic_basis(Z=Z, N=N, n00=nsh, beta=beta, ngh=ngh, ngl=ngl)
    return build_problem(basis, op, K, beta_type, kw.pop("interaction", "SKOP"), **dict(COUPLINGS, **kw))


def rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


def oracle_case(prob, seed):
    from oracle.oracle import Oracle
    orc = Oracle(prob)
    rng = np.random.default_rng(seed)
    rsp, maps = orc.qp_to_sp(*(rng.standard_normal(prob.nxy) for _ in range(4)))
    _, _, xm, ym = orc.fqp()
    fm = prob.f_struct.ir2c
    min_ = np.array([maps[0]] * 2 + [maps[1]] * 2 + [maps[3]] * 2 + [maps[2]] * 2)
    mout = np.array([fm] * 2 + [xm] * 2 + [fm] * 2 + [ym] * 2)
    dens = [orc.densities(rsp[[0, 1, 2, 3]], maps[[0, 0, 1, 1]]), orc.densities(rsp[[6, 7, 4, 5]], maps[[3, 3, 2, 2]])]
    return rsp[ARG], orc.calc_hamiltonian(rsp[ARG], min_, mout), dens


@pytest.mark.parametrize("nsh,ngh,ngl,op,K,kw", [
    (5, 7, 5, "GT", 0, {}), (6, 8, 16, "GT", 1, {}), (6, 9, 17, "F", 0, {}), (7, 16, 31, "R", 1, {}),
    (7, 33, 12, "RS2", 2, {}), (6, 40, 33, "GT", 1, {"beta_type": "+"}), (6, 41, 20, "PS0", 0, {}),
    (5, 65, 6, "GT", 0, {}), (8, 20, 15, "GT", 1, {"beta": 0.3}),
    (6, 17, 14, "GT", 1, {"interaction": "UNEDF2", "override_cds": 3.7, "override_cgs": -2.3, "override_cf": 1.9,
                          "override_csr": 11.0, "override_ct": -5.5, "override_cj": 0.7, "override_csdj": 13.0,
                          "require_gauge_invariance": False}),
])
def test_against_oracle(nsh, ngh, ngl, op, K, kw):
    from pynfam_amd.engine import GpuEngine
    prob = problem(nsh, ngh, ngl, op, K, **kw)
    args, ref_h, ref_d = oracle_case(prob, 7 * nsh + K)
    eng = GpuEngine(prob)
    assert eng.get_option("fp64_separable") == 1
    eng.profile(True)
    got = eng.calc_hamiltonian(args)
    assert any(c.startswith("k_sep_dens<") for c in eng.kernel_classes())
    for k in range(8):
        assert rel(got[k], ref_h[k]) < 1e-12, k
    for sec in (0, 1):
        assert rel(eng.densities(args, sec), ref_d[sec]) < 1e-12, sec
    eng.close()


@pytest.mark.parametrize("npts", [1, 3, 7, 8, 17])
def test_solve_equals_general_kernels(npts):
    """Whole batches, the point counts on either side of the split and tile
    rules: iteration counts equal, strengths as far apart as two FP64 summation
    orders leave them (1e-9, the bar of the oracle's own batches)."""
    from pynfam_amd.engine import GpuEngine
    from pynfam_amd.rate import circle_contour
    prob = problem(8, 22, 19, "GT", 1, Z=60, N=92, beta=0.3)
    w = np.asarray(circle_contour(0.0, 6.0, 2 * npts)["z"][:npts])
    eng = GpuEngine(prob)
    got = eng.solve(w)
    eng.set_option("fp64_grid", 1)
    assert eng.get_option("fp64_separable") == 0
    ref = eng.solve(w)
    eng.close()
    assert np.all(ref["iterations"] > 0) and np.array_equal(got["iterations"], ref["iterations"])
    assert rel(got["strength"], ref["strength"]) < 1e-9


@pytest.mark.parametrize("table", ["wf", "wfdr", "wfdp", "wfdz", "wfd2_all"])
def test_no_product_takes_general_kernels(table):
    """One value of one table off by 1e-9 of the largest: no product any more.
    (The state of the table's largest value: wfdp is zero for Lambda = 0.)"""
    from pynfam_amd.engine import GpuEngine
    prob = problem(6, 14, 13, "GT", 0)
    t = getattr(prob.basis, table).copy(order="F")
    a = int(np.argmax(np.abs(t).max(axis=0)))
    t[17, a] += 1e-9 * np.abs(t[:, a]).max()
    prob = copy.copy(prob)
    prob.basis = copy.copy(prob.basis)
    setattr(prob.basis, table, t)
    args, ref_h, _ = oracle_case(prob, 3)
    eng = GpuEngine(prob)
    assert eng.get_option("fp64_separable") == 0
    got = eng.calc_hamiltonian(args)
    for k in range(8):
        assert rel(got[k], ref_h[k]) < 1e-12, k
    eng.close()


@pytest.mark.parametrize("ngh,ngl,op,K", [(7, 9, "GT", 0), (22, 13, "RS2", 2), (33, 8, "GT", 1), (65, 6, "F", 0)])
@pytest.mark.parametrize("npts", [8, 9, 16, 33])
def test_batch_forms_equal_general_kernels(ngh, ngl, op, K, npts):
    """The forms for a wave, two and four waves per slot, one to three tiles of
    axial points and two groups of them, over two iterations from zero: each
    Hamiltonian agrees to 1e-12 of its largest element (the units' bar), the
    second one's input is the first one's output, hence 1e-11."""
    from pynfam_amd.engine import GpuEngine
    from pynfam_amd.rate import circle_contour
    prob = problem(6, ngh, ngl, op, K)
    w = np.asarray(circle_contour(0.0, 6.0, 2 * npts)["z"][:npts])
    eng = GpuEngine(prob)
    assert eng.get_option("fp64_separable") == 1
    got = eng.solve(w, max_iter=3, want_x=True)
    eng.set_option("fp64_grid", 1)
    ref = eng.solve(w, max_iter=3, want_x=True)
    eng.close()
    assert rel(got["strength"], ref["strength"]) < 1e-11
    assert rel(got["x"], ref["x"]) < 1e-11


@pytest.mark.parametrize("npts,pass_points", [(19, 9), (19, 18), (17, 16), (9, 1), (20, 8)])
@pytest.mark.parametrize("graph", [0, 1])
def test_several_passes(npts, pass_points, graph):
    """A batch in passes of fewer points (option fp64_grid_bytes), the last one of
    another form: the wave, two-wave and four-wave kernels and the projection's
    slot tiles add in the same order, so that without the splits of few points
    the solve has the bits of the one in a single pass; with them (the parts of
    the densities added in another order) amplitudes after two iterations from
    zero differ as those of the general kernels do (1e-11, as above)."""
    from pynfam_amd.engine import GpuEngine
    from pynfam_amd.rate import circle_contour
    prob = problem(6, 22, 13, "GT", 1)
    w = np.asarray(circle_contour(0.0, 6.0, 2 * npts)["z"][:npts])
    eng = GpuEngine(prob)
    eng.set_option("graph", graph)
    for split in (0, 1):
        eng.set_option("few_split", split)
        eng.set_option("fp64_grid_bytes", 0)
        ref = eng.solve(w, max_iter=8 if split == 0 else 3, want_x=True)
        held = eng.get_option("fp64_held_bytes")
        eng.set_option("fp64_grid_bytes", pass_points * eng.get_option("fp64_point_bytes"))
        got = eng.solve(w, max_iter=8 if split == 0 else 3, want_x=True)
        assert eng.get_option("fp64_separable") == 1 and eng.get_option("fp64_held_bytes") < held
        assert np.array_equal(got["iterations"], ref["iterations"])
        if split == 0:
            assert np.array_equal(got["x"], ref["x"]) and np.array_equal(got["strength"], ref["strength"])
        else:
            assert rel(got["x"], ref["x"]) < 1e-11 and rel(got["strength"], ref["strength"]) < 1e-11
    eng.set_option("fp64_grid", 1)
    gen = eng.solve(w, max_iter=3, want_x=True)
    eng.close()
    assert rel(got["x"], gen["x"]) < 1e-11


@pytest.mark.parametrize("ngh,K", [(96, 0), (100, 1), (128, 0)])
def test_dense_axial_grid(ngh, K):
    """Axial points so many that the wavefunctions vanish on the outer half: a few
    states are products with half the points too, the tables are not.  The real
    number is found and the factored results meet the oracle."""
    from pynfam_amd.engine import GpuEngine
    prob = problem(5, ngh, 6, "GT", K)
    args, ref_h, ref_d = oracle_case(prob, 11 + K)
    eng = GpuEngine(prob)
    assert eng.get_option("fp64_separable") == 1
    got = eng.calc_hamiltonian(args)
    for k in range(8):
        assert rel(got[k], ref_h[k]) < 1e-12, k
    for sec in (0, 1):
        assert rel(eng.densities(args, sec), ref_d[sec]) < 1e-12, sec
    eng.close()


def test_small_deviation_takes_general_kernels():
    """A table 2e-14 of its largest value off a product, ten times what the tables'
    own rounding leaves: not replaced by its fit."""
    from pynfam_amd.engine import GpuEngine
    prob = problem(6, 14, 13, "GT", 0)
    eng = GpuEngine(prob)
    assert eng.get_option("fp64_separable") == 1 and 0.0 < eng.get_option("fp64_residual") < 2e-15
    eng.close()
    t = prob.basis.wf.copy(order="F")
    a = int(np.argmax(np.abs(t).max(axis=0)))
    t[17, a] += 2e-14 * np.abs(t[:, a]).max()
    prob = copy.copy(prob)
    prob.basis = copy.copy(prob.basis)
    prob.basis.wf = t
    eng = GpuEngine(prob)
    assert eng.get_option("fp64_separable") == 0
    eng.close()
