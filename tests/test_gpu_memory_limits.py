"""Calls that meet a limit of the device memory: the error is that of the call
that met it, and what can run with less memory runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUPLINGS = dict(vpair_t0=-346.352, override_cs0=128.279, override_csr=0.0, override_cds=0.0)


def problem(nsh=6, ngh=12, ngl=11, op="GT", K=0):
    from pynfam_amd.problem import build_problem
    from pynfam_amd.synthetic import synthetic_basis
    return build_problem(synthetic_basis(Z=20, N=28, n00=nsh, beta=0.0, ngh=ngh, ngl=ngl), op, K, "-", "SKOP",
                         **COUPLINGS)


def contour(npts):
    from pynfam_amd.rate import circle_contour
    return np.asarray(circle_contour(0.0, 6.0, 2 * npts)["z"][:npts])


def test_failed_allocation_is_reported_once():
    """A batch that no device holds (its first buffer alone takes 512 GB) is
    refused for want of memory; the calls after it run as before."""
    from pynfam_amd.engine import GpuEngine
    eng = GpuEngine(problem())
    w = contour(3)
    ref = eng.solve(w)
    n = int(512e9 / (4 * eng.nxy * 8))
    with pytest.raises(RuntimeError, match="hipMalloc of"):
        eng.solve(np.full(n, 1.0 + 1.0j))
    got = eng.solve(w)
    assert np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(got["strength"], ref["strength"])
    eng.close()


@pytest.mark.parametrize("graph", [0, 1])
def test_no_memory_for_the_factored_stage(graph):
    """A limit below one point's intermediates: solves and per-unit calls give
    the bits of the kernels over all grid points, and nothing is held; without
    the limit both take the factored stage again."""
    from pynfam_amd.engine import GpuEngine
    eng = GpuEngine(problem(K=1))
    args = np.random.default_rng(2).standard_normal((8, eng.nxy))
    eng.set_option("graph", graph)
    w = contour(5)
    first, unit = eng.solve(w), eng.calc_hamiltonian(args)
    assert eng.get_option("fp64_separable") == 1 and eng.get_option("fp64_held_bytes") > 0
    eng.set_option("fp64_grid_bytes", eng.get_option("fp64_point_bytes") - 1)
    eng.profile(True)
    got_unit = eng.calc_hamiltonian(args)
    classes = eng.kernel_classes()
    eng.profile(False)
    assert not any(c.startswith("k_sep_") for c in classes), sorted(classes)
    got = eng.solve(w)
    assert eng.get_option("fp64_separable") == 0 and eng.get_option("fp64_held_bytes") == 0
    eng.set_option("fp64_grid", 1)
    ref, ref_unit = eng.solve(w), eng.calc_hamiltonian(args)
    assert np.array_equal(got["strength"], ref["strength"]) and np.array_equal(got["iterations"], ref["iterations"])
    assert np.array_equal(got_unit, ref_unit)
    eng.set_option("fp64_grid", 0)
    # a call that lacked the memory does not bind the ones after it
    assert np.array_equal(eng.solve(w)["strength"], got["strength"])
    eng.set_option("fp64_grid_bytes", 0)
    assert np.array_equal(eng.calc_hamiltonian(args), unit)
    assert np.array_equal(eng.solve(w)["strength"], first["strength"])
    assert eng.get_option("fp64_separable") == 1
    eng.close()


def test_batch_takes_the_memory_of_the_factored_stage():
    """A batch that cannot be allocated gets what the stage holds before it is
    refused."""
    from pynfam_amd.engine import GpuEngine
    eng = GpuEngine(problem())
    w = contour(3)
    ref = eng.solve(w)
    assert eng.get_option("fp64_held_bytes") > 0
    with pytest.raises(RuntimeError, match="hipMalloc of"):
        eng.solve(np.full(int(512e9 / (4 * eng.nxy * 8)), 1.0 + 1.0j))
    assert eng.get_option("fp64_held_bytes") == 0
    assert np.array_equal(eng.solve(w)["strength"], ref["strength"])
    eng.close()
