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


@pytest.mark.parametrize("nsh,K,beta", [(6, 0, 0.0), (16, 1, 0.3)])
def test_form_by_points(nsh, K, beta):
    """Up to four points one launch of the split form, over the widest class of a
    stage; beyond, a launch per column class, four waves to a workgroup or two
    where four would leave two or three idle.  No other form runs."""
    from pynfam_amd.engine import GpuEngine
    from pynfam_amd.problem import build_problem
    from pynfam_amd.synthetic import synthetic_basis
    prob = build_problem(synthetic_basis(Z=20, N=28, n00=nsh, beta=beta, ngh=8, ngl=6), "GT", K, "-")
    db = np.asarray(prob.basis.db)
    eng = GpuEngine(prob)
    maps, xy = eng.structures()
    rng = np.random.default_rng(6)
    x, hsp = [rng.standard_normal(prob.nxy) for _ in range(4)], rng.standard_normal((8, prob.nxy))
    for reps in (1, 4, 5, 9):
        eng.set_option("unit_replicas", reps)
        for call, blocks in ((lambda: eng.qp2sp(*x), maps), (lambda: eng.sp2qp(hsp), xy)):
            strips = {}   # column class -> strips of its tallest block
            for m in blocks:
                for i, j in enumerate(m):
                    if j >= 0:
                        c = (int(db[j]) + 15) // 16
                        strips[c] = max(strips.get(c, 0), (int(db[i]) + 15) // 16)
            if reps <= 4:
                want = {f"k_triprod_split<{max(strips)}>"}
            else:
                want = {f"k_triprod_mfma<{c},{4 if s % 4 in (0, 3) else 2}>" for c, s in strips.items()}
            eng.profile(True)
            call()
            got = {c for c in eng.kernel_classes() if c.startswith("k_triprod_split") or "," in c}
            eng.profile(False)
            assert got == want, (reps, sorted(got), sorted(want))
    eng.close()
