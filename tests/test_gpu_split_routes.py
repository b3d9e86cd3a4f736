"""The split step's own tests, on the split step.  Plans whose tile nobody sets take the resident
loop where it is faster, so tests that were written for the split kernels (their parity with the
oracle, banded workgroup orders, several rounds of reverse-step workgroups) run here once more with
tiles of 8 rows."""
import pytest

import test_gpu_discrete as discrete
import test_gpu_edges as edges
import test_gpu_fused as fused
import test_gpu_parity as parity
from cuda_fwi_amd import psvfwi as P

pytestmark = pytest.mark.gpu

RUNS = [(parity, "test_forward_bit_exact", dict(case=c, prec=p)) for c in parity.CASES for p in ("fp64", "fp32")]
RUNS += [(parity, "test_gradient_fp64_bit_exact", dict(fdorder=o, win=w)) for o in (2, 4) for w in parity.WINDOWS]
RUNS += [(parity, "test_gradient_fp32_bit_exact_and_tolerance", dict(fdorder=o)) for o in (2, 4)]
RUNS += [(parity, "test_checkpoint_gradient_equals_full_store", dict(prec=p)) for p in ("fp64", "fp32")]
RUNS += [(parity, t, {}) for t in ("test_batched_uneven_shots_equal_single_shots",
                                   "test_explosive_and_vx_sources_bit_exact",
                                   "test_colocated_sources_and_boundary_geometry")]
RUNS += [(edges, t, {}) for t in ("test_batch_with_a_shot_without_receivers_and_one_without_sources",
                                  "test_empty_window_gives_zero_store_and_gradient")]
RUNS += [(fused, "test_shot_orders_give_identical_results", {}),
         (discrete, "test_discrete_gradient_batched_uneven_shots", dict(segment=33)),
         (discrete, "test_discrete_gradient_many_workgroups", {})]


@pytest.mark.parametrize("module,name,args", RUNS, ids=lambda v: getattr(v, "__name__", None) or
                         ("-".join(map(str, v.values())) if isinstance(v, dict) else v))
def test_on_the_split_step(module, name, args, monkeypatch):
    plans, plan_of = [], module.plan_of

    def split(pb, precision="fp64", tz=None, shots=None):
        plans.append(plan_of(pb, precision, tz=tz or 8, shots=shots))
        return plans[-1]

    monkeypatch.setattr(module, "plan_of", split)
    autotune, tuned = P.Plan.autotune, []
    monkeypatch.setattr(P.Plan, "autotune", lambda p, *a: (tuned.append(p), autotune(p, *a))[1])
    getattr(module, name)(**args)
    assert plans
    for p in plans:
        if p not in tuned and p._h:
            assert p.last_step("forward") == (8, False)
            p.close()
