"""The Broyden hook at history lengths on either side of the dots kernel's passes of
eight vectors, at one entry and at the most the engine holds, past the wrap of
each, against the oracle's Broyden.

Both sides solve the same small linear system from dot products of a few
thousand FP64 terms (1e-15 each).  For random residuals the normalised
differences' Gram matrix is close to tridiagonal (-1/2, 1, -1/2), of condition
2e3 at 64 entries: 1e-11 of the largest element, the bar of the hook's other
test."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 7, 8, 9, 16, 17, 30, 64])
def test_history_lengths_against_oracle(M):
    from oracle.oracle import Broyden
    from pynfam_amd.engine import GpuEngine
    from test_gpu_separable import problem
    eng = GpuEngine(problem(6, 8, 6))
    n = 4 * eng.nxy
    ob = Broyden(n, M)
    rng = np.random.default_rng(M)
    vin = np.zeros(n)
    for it in range(M + 4):
        vout = vin + rng.standard_normal(n)
        rg, vg, si_g, _ = eng.broyden_step(it, vout, vin, broyden_history=M)
        ro, vo, si_o, _ = ob.step(it, vout, vin)
        assert abs(si_g - si_o) <= 1e-14 * si_o
        assert np.max(np.abs(rg - ro)) <= 1e-14 * np.max(np.abs(ro))
        assert np.max(np.abs(vg - vo)) <= 1e-11 * np.max(np.abs(vo)), it
        vin = vg   # both go on from the same vector
    eng.close()
