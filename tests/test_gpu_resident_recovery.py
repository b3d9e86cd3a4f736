"""The resident loop's way out: a wait that gives up or a launch that is refused (both forced from
the host: every kernel still ends by itself) has the run done again with the split step, bit for
bit, and the exchange's tags may run over."""
import time

import numpy as np
import pytest

import refcase as RC
from gpucase import plan_of
from test_gpu_resident import _problem, _same

pytestmark = pytest.mark.gpu

# nx, nz, npml, order, fsurf, precision, nt, K: several tiles; strips
GRIDS = [(101, 77, 8, 4, 1, "fp32", 60, 1.0), (160, 120, 10, 2, 0, "fp64", 45, 1.0), (1900, 700, 20, 4, 0, "fp32", 70, 1.0)]
FORCE = {"wait": dict(mute=1), "refused": dict(refuse=1)}


def _setup(plan, mode):
    if mode == "discrete":
        plan.set_gradient_mode("discrete", 31)
    else:
        plan.set_store_mode(mode, 29)


def _forward(plan):
    plan.forward(energy=True, gradient=True)
    return [plan.records(i) for i in range(2)] + [plan.field("We", i) for i in range(2)]


def _adjoint(plan, mode, obs):
    plan.misfit(obs)
    plan.adjoint(energy=True, gradient=True)
    if mode == "discrete":
        return list(plan.model_gradient())
    return list(plan.gradient()) + [plan.field("We", i) for i in range(2)]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda c: f"{c[0]}x{c[1]}{c[5]}")
@pytest.mark.parametrize("mode", ["full", "checkpoint", "discrete"])
@pytest.mark.parametrize("how", list(FORCE))
def test_run_is_done_again(grid, mode, how):
    print(f"done again {grid} {mode} {how}", flush=True)
    pb, shots, obs = _problem(grid, 2, dict(dt=2))
    ref, plan = (plan_of(pb, grid[5], tz=tz, shots=shots) for tz in (8, None))
    for p in (ref, plan):
        _setup(p, mode)
    f, a = _forward(ref), _adjoint(ref, mode, obs)
    plan.test_resident(**FORCE[how])
    assert all(_same(x, y) for x, y in zip(_forward(plan), f))
    assert plan.last_step("forward") == (8, True)
    plan.test_resident()
    assert all(_same(x, y) for x, y in zip(_adjoint(plan, mode, obs), a))
    assert plan.last_step("adjoint") == (8, True)
    # asked for again: the forward runs resident, and then the adjoint gives up
    plan.set_tile(0)
    assert all(_same(x, y) for x, y in zip(_forward(plan), f))
    assert plan.last_step("forward") == (0, False)
    plan.test_resident(**FORCE[how])
    assert all(_same(x, y) for x, y in zip(_adjoint(plan, mode, obs), a))
    assert plan.last_step("adjoint") == (8, True)
    plan.set_tile(0)
    plan.test_resident()
    _forward(plan)
    assert all(_same(x, y) for x, y in zip(_adjoint(plan, mode, obs), a))
    assert plan.last_step("adjoint") == (0, False)
    ref.close()
    plan.close()


def test_wait_runs_out():
    """Nobody ends the wait but its own count of tries: long enough for kernels of other processes to
    leave the GPU, and no more than a few seconds."""
    print("wait runs out", flush=True)
    pb, shots, obs = _problem(GRIDS[0], 2, dict(dt=2))
    ref, plan = (plan_of(pb, "fp32", tz=tz, shots=shots) for tz in (8, None))
    _forward(plan)
    plan.test_resident(mute=2)
    t = time.perf_counter()
    r = _forward(plan)
    t = time.perf_counter() - t
    assert all(_same(x, y) for x, y in zip(r, _forward(ref)))
    assert plan.last_step("forward") == (8, True)
    assert 1.0 < t < 6.0, t
    ref.close()
    plan.close()


@pytest.mark.parametrize("how", list(FORCE))
def test_autotuner_without_the_loop(how):
    print(f"autotuner {how}", flush=True)
    pb = RC.small_problem(nx=101, nz=77, npml=8, nt=60, fdorder=4)
    plan = plan_of(pb, "fp32")
    plan.test_resident(**FORCE[how])
    best = plan.autotune(10)
    plan.test_resident()
    plan.forward()
    assert plan.last_step("forward") == (best, True)
    plan.close()


@pytest.mark.parametrize("grid", GRIDS, ids=lambda c: f"{c[0]}x{c[1]}{c[5]}")
def test_exchange_tags_run_over(grid):
    print(f"tags run over {grid}", flush=True)
    pb, shots, obs = _problem(grid, 2, dict(dt=2))
    ref, plan = (plan_of(pb, grid[5], tz=tz, shots=shots) for tz in (8, None))
    plan.forward()
    f, a = _forward(ref), _adjoint(ref, "full", obs)
    # the last launch before the fill, and every place of it in the runs
    for left in (3, grid[6] + 1, grid[6] + 2, grid[6] + 3, 3 * grid[6]):
        plan.test_resident(tag=0xffffffff - left)
        assert all(_same(x, y) for x, y in zip(_forward(plan), f)), left
        assert all(_same(x, y) for x, y in zip(_adjoint(plan, "full", obs), a)), left
        assert plan.last_step("forward") == plan.last_step("adjoint") == (0, False)
    ref.close()
    plan.close()
