"""Which step a run takes: the resident time loop or the step kernels, and that every caller's
route gives the split step's results bit for bit."""
import numpy as np
import pytest

import psv_oracle as O
import refcase as RC
from cuda_fwi_amd import psvfwi as P
from gpucase import plan_of, shots_of
from test_gpu_resident import CASES, _problem, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}p{c[2]}o{c[3]}fs{c[4]}{c[5]}K{c[7]}")
def test_exact_gradient_takes_the_resident_loop(case):
    """The replay and the transposed steps of every shape are built and chosen: what the equality
    with the split step is about."""
    print(f"route of the exact gradient {case}", flush=True)
    pb, shots, obs = _problem(case, 2, dict(dt=1))
    plan = plan_of(pb, case[5], shots=shots)
    plan.set_gradient_mode("discrete", max(8, case[6] // 2 - 3))
    plan.forward(gradient=True)
    plan.misfit(obs)
    plan.adjoint(gradient=True)
    assert plan.last_step("forward") == (0, False)
    assert plan.last_step("adjoint") == (0, False)
    plan.close()


def test_last_step_names_the_step():
    print("last step", flush=True)
    pb = RC.small_problem(nx=60, nz=40, npml=8, nt=40, fdorder=4)
    plan = plan_of(pb, "fp32", tz=-16)
    with pytest.raises(P.PsvfwiError) as e:
        plan.last_step("forward")
    assert e.value.status == -5
    for tz in (-16, 4, 0):
        plan.set_tile(tz)
        plan.forward()
        assert plan.last_step("forward") == (tz, False)
    with pytest.raises(P.PsvfwiError):
        plan.last_step("adjoint")
    plan.close()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_rounds_of_several_shots(prec):
    """More shots than one launch holds: rounds of several shots, the last one not full, records
    of uneven length."""
    print(f"rounds of shots {prec}", flush=True)
    base = RC.small_problem(nx=200, nz=100, npml=40, nt=10, fdorder=4, fsurf=0, hetero=True)
    shots, obs = [], []
    rng = np.random.default_rng(8)
    for i in range(19):
        nt = 40 + 3 * (i * 7 % 19)
        sig = O.create_wavelet(nt, base.dt, 1.0 + i, 25.0, 0.0)[None]
        shots.append(dict(nt=nt, src=dict(x=[60 + 9 * i], z=[base.ppad + 4 + i], comp=[2]), src_signal=sig,
                          rec=dict(x=[58 + 9 * i, 140, 150], z=[base.ppad + 3 + i] * 3, comp=[2, 1, 2])))
        obs.append(rng.standard_normal((3, nt)) * 1e-3)
    out = []
    for tz in (8, None):
        plan = plan_of(base, prec, tz=tz, shots=shots)
        r = []
        for mode in (("full", 0), ("checkpoint", 17), "discrete"):
            plan.set_window(RC.full_window(base, dt=2))
            if mode == "discrete":
                plan.set_gradient_mode("discrete", 30)
            else:
                plan.set_store_mode(*mode)
            plan.forward(gradient=True)
            r += [plan.records(i) for i in range(19)] + [plan.misfit(obs)]
            plan.adjoint(gradient=True)
            r += list(plan.model_gradient(-1) if mode == "discrete" else plan.gradient(-1))
            for kind in ("forward", "adjoint"):
                assert plan.last_step(kind) == (tz or 0, False)
        plan.close()
        out.append(r)
    assert all(np.abs(a).max() > 0 for a in out[0])
    assert all(_same(a, b) for a, b in zip(*out))


def test_autotuned_tile_serves_the_runs_the_loop_cannot():
    """On 88 x 88 cells tiles of 8 rows are never the fastest: on the GPU those of 4 are a quarter
    faster, and where the host's launches set the pace the fused step with one a step is.  The
    autotuner returns what it measured, and what cannot run resident (snapshots, short checkpoint
    intervals, the random-boundary adjoint) takes the fastest split tile."""
    print("autotuned tile beside the resident loop", flush=True)
    pb = RC.small_problem(nx=84, nz=84, npml=0, nt=60, fdorder=4, fsurf=0, nrec=6)
    pb.lam, pb.mu, pb.rho = P.random_boundary(pb.lam, pb.mu, pb.rho, 12, 0, seed=5, max_increase=0.3)
    pb.mu_zx, pb.rho_zp, pb.rho_xp = O.average_parameters(pb.mu, pb.rho)
    pb.fwi = RC.full_window(pb, dt=2)
    obs = [1e-3 * np.random.default_rng(2).standard_normal((6, pb.nt))]
    plan = plan_of(pb, "fp64")
    best = plan.autotune(40)
    assert best in (4, 16, -8, -16)
    plan.forward()
    assert plan.last_step("forward") == (0, False)
    plan.set_snapshots(10)
    plan.forward()
    split = plan.last_step("forward")
    assert split[0] in ((best,) if best > 0 else (4, 8, 16)) and not split[1]
    plan.set_snapshots(0)
    plan.set_store_mode("checkpoint", 4)
    plan.forward(gradient=True)
    plan.misfit(obs)
    plan.adjoint()
    assert plan.last_step("forward") == plan.last_step("adjoint") == split
    g = plan.gradient()
    ref = plan_of(pb, "fp64", tz=8)
    for p in (plan, ref):
        p.set_store_mode("random_boundary")
        p.forward(gradient=True)
        p.misfit(obs)
        p.adjoint()
    assert plan.last_step("adjoint") == split
    assert all(_same(a, b) for a, b in zip(plan.gradient(), ref.gradient()))
    ref.set_store_mode("full")
    ref.forward(gradient=True)
    ref.misfit(obs)
    ref.adjoint()
    assert all(_same(a, b) for a, b in zip(g, ref.gradient()))


@pytest.mark.parametrize("grid,segments,short,long", [((84, 84, 0, 4, 0, "fp64"), False, 2, 16),
                                                      ((1900, 700, 20, 4, 0, "fp32"), False, 4, 16),
                                                      ((2400, 800, 20, 4, 1, "fp64"), True, 8, 32)],
                         ids=lambda g: "x".join(map(str, g)) if isinstance(g, tuple) else str(g))
def test_short_runs_stay_on_the_split_step(grid, segments, short, long):
    """A resident launch loads and writes the whole state: records of a step or two, and on grids in
    strips of a few steps, and segments of 8 there, are faster on the split step.  Either way the same
    results."""
    print(f"short runs {grid}", flush=True)
    pb, shots, obs = _problem(grid + (48, 1.0), 2, dict(dt=2))
    for k in (short, long):
        nt = pb.nt if segments else k
        one = dict(shots[0], nt=nt, src_signal=shots[0]["src_signal"][:, :nt])
        out = []
        for tz in (8, None):
            plan = plan_of(pb, grid[5], tz=tz, shots=[one])
            plan.set_store_mode("checkpoint" if segments else "full", k)
            plan.forward(gradient=True)
            r = [plan.records(), plan.misfit([obs[0][:, :nt]])]
            plan.adjoint()
            out.append(r + list(plan.gradient()))
            want = 8 if tz or k == short else 0
            assert [plan.last_step(q)[0] for q in ("forward", "adjoint")] == [want, want], k
            plan.close()
        assert all(_same(a, b) for a, b in zip(*out))


def test_timing_holds_no_host_work():
    """The run's time (HIP events) is that of its steps: the point tables of a new batch, more than a
    millisecond of host work here, are made before it starts."""
    print("timing of the first run of a batch", flush=True)
    pb = RC.small_problem(nx=1000, nz=500, npml=40, nt=16, fdorder=4, hetero=False)
    rec = dict(x=[45 + 2 * i for i in range(400)], z=[pb.ppad + i % 3 for i in range(400)], comp=[2] * 400)
    shots = [dict(shots_of(pb), rec=rec) for _ in range(24)]
    plan = plan_of(pb, "fp32", shots=shots)
    first, again = [], []
    for _ in range(4):
        plan.set_shots(shots)
        for ms in (first, again):
            plan.forward(energy=False)
            ms.append(plan.timing()[0])
    assert plan.last_step("forward") == (0, False)
    plan.close()
    assert min(first) < 1.25 * min(again), (first, again)


def test_large_fp64_adjoint_stays_on_the_split_step():
    """2000 x 4000 cells need the largest FP64 tiles, whose adjoint step with the correlation spills
    registers: 459 us a step against 353 of the split step; forward 244 against 298."""
    print("large FP64 grid", flush=True)
    pb = RC.small_problem(nx=2000, nz=4000, npml=40, nt=64, fdorder=4, fsurf=0, hetero=False)
    pb.fwi = dict(dt=4, dx=1, dz=1, x1=600, x2=900, z1=42, z2=200)
    obs = [1e-3 * np.random.default_rng(5).standard_normal((5, pb.nt))]
    out = []
    for tz in (8, None):
        plan = plan_of(pb, "fp64", tz=tz)
        plan.forward(gradient=True)
        r = [plan.records(), plan.misfit(obs)]
        plan.adjoint(energy=False)
        out.append(r + list(plan.gradient()))
        assert [plan.last_step(k)[0] for k in ("forward", "adjoint")] == [tz or 0, 8]
        if tz:
            plan.close()
    assert all(_same(a, b) for a, b in zip(*out))
    # its exact gradient: segments of 8 steps 1490 us a step in the loop and 1110 split, of 32 1000 and 1070
    out = []
    for k, want in ((8, 8), (32, 0)):
        plan.set_gradient_mode("discrete", k)
        plan.forward(energy=False, gradient=True)
        plan.misfit(obs)
        plan.adjoint(energy=False)
        assert plan.last_step("adjoint") == (want, False)
        out.append(plan.model_gradient())
    plan.close()
    assert all(_same(a, b) for a, b in zip(*out))
