"""Several plans on one GPU at the same time, one per host thread: two resident loops and a split
step.  Launches of the resident loop take the GPU one after another; the results of each plan are
those it has alone, bit for bit, and none gives the loop up."""
import threading

import numpy as np
import pytest

from gpucase import plan_of
from test_gpu_resident import _problem, _same

pytestmark = pytest.mark.gpu

# the last one with tiles of 8 rows, in two launches a step
GRIDS = [((420, 300, 20, 4, 1, "fp32", 200, 1.0), None), ((160, 120, 10, 2, 0, "fp64", 200, 1.0), None),
         ((250, 180, 12, 4, 0, "fp32", 200, 1.0), 8)]


def _pass(plan, obs, discrete):
    plan.set_gradient_mode("discrete" if discrete else "reference", 50)
    plan.forward(energy=True, gradient=True)
    r = [plan.records(i) for i in range(2)] + [plan.misfit(obs)]
    plan.adjoint(gradient=True)
    return r + list(plan.model_gradient() if discrete else plan.gradient())


def test_plans_side_by_side():
    print("plans side by side", flush=True)
    made = []
    for grid, tz in GRIDS:
        pb, shots, obs = _problem(grid, 2, dict(dt=2))
        plan = plan_of(pb, grid[5], tz=tz, shots=shots)
        made.append((plan, obs, tz, [_pass(plan, obs, d) for d in (False, True)]))
    bad = []

    def work(k):
        try:
            plan, obs, tz, ref = made[k]
            for i in range(12):
                r = _pass(plan, obs, i % 2 == 1)
                if not all(_same(a, b) for a, b in zip(r, ref[i % 2])):
                    bad.append((k, i))
                if any(plan.last_step(kind) != (tz or 0, False) for kind in ("forward", "adjoint")):
                    bad.append((k, i, plan.last_step("forward"), plan.last_step("adjoint")))
        except Exception as e:  # a thread's exception would not fail the test
            bad.append((k, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(made))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for plan, *_ in made:
        plan.close()
    assert not bad, bad
