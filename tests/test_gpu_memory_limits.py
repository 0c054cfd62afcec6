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
