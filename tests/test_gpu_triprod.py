"""FP64 block triple products (both transforms) at the edges of their tiles and
dispatch: block sizes below, at and above the 16-column tiles, all eight column
classes, groups of one to eight strips (two or four waves per workgroup), and the
numbers of points on either side of the one-launch form, against the oracle.

The bar is that of the other FP64 units, 1e-12 of each array's largest element
(sums of a few hundred FP64 terms, some 1e-15 each)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ARG = [0, 1, 2, 3, 6, 7, 4, 5]   # quadrant slots <-> calc_dHsp_interface argument order


def rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


@pytest.mark.parametrize("nsh,op,K,beta", [(2, "GT", 0, 0.0), (6, "RS2", 2, 0.0), (8, "F", 0, 0.0), (10, "R", 1, 0.0),
                                           (14, "GT", 1, 0.3), (16, "GT", 0, 0.0), (18, "GT", 1, 0.0),
                                           (20, "RS2", 2, 0.0)])
def test_transforms_at_tile_edges(nsh, op, K, beta):
    from oracle.oracle import Oracle
    from pynfam_amd.engine import GpuEngine
    from pynfam_amd.problem import build_problem
    from pynfam_amd.synthetic import synthetic_basis
    prob = build_problem(synthetic_basis(Z=20, N=28, n00=nsh, beta=beta, ngh=8, ngl=6), op, K, "-")
    orc = Oracle(prob)
    rng = np.random.default_rng(40 + nsh + K)
    x = [rng.standard_normal(prob.nxy) for _ in range(4)]
    ref, _ = orc.qp_to_sp(*x)
    hsp = rng.standard_normal((8, prob.nxy))
    _, _, xm, ym = orc.fqp()
    fm = prob.f_struct.ir2c
    ref_q = orc.sp_to_qp(hsp[ARG], np.array([fm, xm, ym, fm]))
    eng = GpuEngine(prob)
    for reps in (1, 4, 5, 9):
        eng.set_option("unit_replicas", reps)
        print(f"[n00={nsh} K={K} beta={beta} replicas={reps}]", flush=True)
        assert rel(eng.qp2sp(*x), ref) < 1e-12, reps
        got = eng.sp2qp(hsp)
        for k in range(4):
            assert rel(got[k], ref_q[k]) < 1e-12, (reps, k)
    eng.close()
