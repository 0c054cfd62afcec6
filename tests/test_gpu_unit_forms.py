"""Which form of the FP64 grid stage the per-unit calls take, and the factored
form of it at the configuration sizes.

`unit_replicas` alone leaves the per-unit calls on the kernels over all grid
points (the other configuration tests use that); `unit_general` 0 afterwards
gives them the form the solves take.  The factored stage is then compared with
the oracle at the sizes and with the bar of the other FP64 units (1e-12 of each
array's largest element), for one point, for 12 (two waves per slot) and for 17
(four waves per slot)."""
import numpy as np
import pytest

from conftest import golden_problem
from test_gpu_config_sizes import ARG, case, rel   # noqa: F401  (case is a fixture)

pytestmark = pytest.mark.gpu


def unit_classes(eng, args):
    eng.profile(True)
    out = eng.calc_hamiltonian(args)
    got = eng.kernel_classes()
    eng.profile(False)
    return out, any(c.startswith("k_sep_dens<") for c in got)


def test_tuning_leaves_the_unit_calls_as_they_were(tmp_path, monkeypatch):
    from pynfam_amd import autotune
    from pynfam_amd.engine import GpuEngine
    monkeypatch.setenv("PNFAM_GPU_TUNE_CACHE", str(tmp_path / "tune.json"))
    eng = GpuEngine(golden_problem("S40", 0))
    args = np.random.default_rng(4).standard_normal((8, eng.nxy))
    before, factored = unit_classes(eng, args)
    assert factored
    assert not autotune.tune(eng, batch=4, repeats=1)["cached"]
    after, factored = unit_classes(eng, args)
    assert factored and np.array_equal(before, after)
    eng.close()


def test_replicas_leave_a_way_back():
    from pynfam_amd.engine import GpuEngine
    eng = GpuEngine(golden_problem("S40", 1))
    args = np.random.default_rng(5).standard_normal((8, eng.nxy))
    first, factored = unit_classes(eng, args)
    assert factored and eng.get_option("unit_general") == 0
    eng.set_option("unit_replicas", 1)
    assert eng.get_option("unit_general") == 1 and not unit_classes(eng, args)[1]
    eng.set_option("unit_general", 0)
    again, factored = unit_classes(eng, args)
    assert factored and np.array_equal(first, again)
    eng.set_option("fp64_grid", 1)
    assert not unit_classes(eng, args)[1]
    eng.close()


@pytest.mark.parametrize("reps", [1, 12, 17])
def test_factored_units_against_oracle(case, reps):   # noqa: F811
    from pynfam_amd.engine import GpuEngine
    print(f"[{case['cfg']} K={case['K']} replicas={reps}] factored FP64 units", flush=True)
    eng = GpuEngine(case["prob"])
    eng.set_option("unit_replicas", reps)
    eng.set_option("unit_general", 0)
    eng.profile(True)
    got = eng.calc_hamiltonian(case["rsp"][ARG])
    for k in range(8):
        assert rel(got[k], case["ref_h"][k]) < 1e-12, k
    for sec in (0, 1):
        assert rel(eng.densities(case["rsp"][ARG], sec), case["ref_d"][sec]) < 1e-12, sec
    launched = eng.kernel_classes()
    forms = {1: {"k_sep_z", "k_sep_expand"}, 12: {"k_sep_z_wide<2>", "k_sep_expand_wide<2>"},
             17: {"k_sep_z_wide<4>", "k_sep_expand_wide<4>"}}[reps]
    assert forms <= launched and any(c.startswith("k_sep_proj<") for c in launched), sorted(launched)
    assert not any(c.startswith(("k_density", "k_project")) for c in launched), sorted(launched)
    eng.close()
