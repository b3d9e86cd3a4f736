"""The resident time loop (the automatic choice where a grid fits: many steps per launch, the
wavefields in registers, tiles that exchange their rims) against the split step kernels, which
the oracle's tests pin: records, wavefields, CPML memory, illumination and both gradients, bit
for bit, at the sizes where a tile can go wrong: the smallest grid, one tile to three columns of
them, every tile shape of the three types, both orders, the free surface, no CPML, K != 1,
checkpoint segments with a short last one, grids in strips, uneven shots, sources of every kind, a strided window."""
import numpy as np
import pytest

import psv_oracle as O
import refcase as RC
from gpucase import plan_of, shots_of
from test_gpu_parity import MEMS

pytestmark = pytest.mark.gpu

# nx, nz, npml, order, fsurf, precision, nt, K at the outer edge
CASES = [
    (12, 12, 0, 4, 0, "fp32", 60, 1.0),        # 16 x 16: the smallest
    (14, 14, 0, 2, 1, "fp64", 60, 1.0),
    (52, 60, 4, 4, 0, "fp32", 150, 1.5),       # 64 columns: one column of tiles
    (53, 41, 4, 4, 1, "fp32", 150, 1.0),       # 65: two
    (100, 30, 8, 2, 1, "fp32", 150, 1.0),      # 118
    (101, 77, 8, 4, 1, "fp32", 150, 1.5),      # 121: three
    (101, 77, 8, 4, 0, "fp64", 150, 1.0),
    (160, 120, 10, 2, 0, "fp64", 60, 1.5),
    (90, 70, 8, 4, 1, "fp32x2", 60, 1.5),
    (250, 180, 12, 4, 0, "fp32x2", 24, 1.0),
    (380, 240, 20, 4, 1, "fp64", 24, 1.0),
    (560, 380, 20, 4, 1, "fp64", 24, 1.0),
    (420, 300, 20, 4, 1, "fp32", 40, 1.0),
    (760, 520, 30, 2, 1, "fp32", 40, 1.0),
    (1000, 500, 40, 4, 0, "fp32", 40, 1.0),
    (1400, 600, 40, 4, 1, "fp32", 24, 1.0),
    (1900, 700, 20, 4, 1, "fp32", 45, 1.5),    # strips; the last segment is one step
    (1000, 600, 20, 2, 0, "fp64", 45, 1.0),
]


def _problem(case, comp, window):
    nx, nz, npml, order, fsurf, prec, nt, kmax = case
    pb = RC.small_problem(nx=nx, nz=nz, npml=npml, nt=nt, fsurf=fsurf, fdorder=order, seed=nx, nrec=7, src_comp=comp)
    pb.pml = O.cpml_pro(npml, 5.0, 25.0, 2.0, kmax, 1e-3, 2750.0, 5e-4)
    pb.fwi = RC.full_window(pb, **window)
    # receivers and sources of both components, some in one cell, some at the seams of tiles
    pb.rec["comp"] = [1, 2, 2, 1, 2, 1, 2]
    pb.rec["x"][0] = pb.src["x"][0] + 1   # near a source: the gradients are not zero
    pb.rec["x"][3] = pb.rec["x"][2]
    pb.rec["x"][4] = min(56, pb.nxt - 4)
    pb.rec["z"][4] = pb.nzt // 2
    pb.src["x"][1] = min(59, pb.nxt - 4)
    a, b = shots_of(pb), shots_of(pb)
    b["nt"] = nt - nt // 3
    b["src_signal"] = a["src_signal"][:, :b["nt"]] * 0.5
    obs = [1e-3 * np.random.default_rng(i).standard_normal((7, s["nt"])) for i, s in enumerate((a, b))]
    return pb, [a, b], obs


def _same(x, y):
    return np.array_equal(np.asarray(x), np.asarray(y))


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}p{c[2]}o{c[3]}fs{c[4]}{c[5]}K{c[7]}")
def test_resident_equals_split_step(case):
    print(f"resident {case}", flush=True)
    nt, prec = case[6], case[5]
    for comp, window, mode in ((2, dict(dt=2), ("full", 0)), (4, dict(dt=3, dx=2, dz=3), ("checkpoint", (nt - 1) // 2))):
        pb, shots, obs = _problem(case, comp, window)
        out = []
        for tz in (8, None):
            plan = plan_of(pb, prec, tz=tz, shots=shots)
            plan.set_store_mode(*mode)
            plan.set_observed(obs)
            plan.forward(energy=True, gradient=True)
            # one kernel per run of steps (the split step times two)
            assert (plan.kernel_timing("forward")[1] == 0) == (tz is None)
            r = [plan.records(i) for i in range(2)] + [plan.field("We", i) for i in range(2)]
            names = ["vx", "vz", "sxx", "szx", "szz"] + list(MEMS if case[2] else ())
            r += [plan.field(k, i) for k in names for i in range(2)]
            r.append(plan.misfit())
            plan.adjoint(energy=True, gradient=True)
            r += [plan.field(k, i) for k in names + ["ux", "uz", "We"] for i in range(2)]
            r += [g for i in range(2) for g in plan.gradient(i)]
            plan.close()
            out.append(r)
        assert all(_same(a, b) for a, b in zip(*out)), [k for k, (a, b) in enumerate(zip(*out)) if not _same(a, b)]
        assert np.abs(out[0][-3]).max() > 0


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}x{c[1]}p{c[2]}o{c[3]}fs{c[4]}{c[5]}K{c[7]}")
def test_resident_exact_gradient_equals_split_step(case):
    print(f"resident exact gradient {case}", flush=True)
    pb, shots, obs = _problem(case, 2, dict(dt=1))
    out = []
    for tz in (8, None):
        plan = plan_of(pb, case[5], tz=tz, shots=shots)
        plan.set_gradient_mode("discrete", max(8, case[6] // 2 - 3))
        plan.set_observed(obs)
        plan.forward(gradient=True)
        plan.misfit()
        plan.adjoint(gradient=True)
        out.append([plan.coefficient_gradient(i) for i in range(2)])
        plan.close()
    for i in range(2):
        for k in out[0][i]:
            assert np.abs(out[0][i][k]).max() > 0, k
            assert np.array_equal(out[0][i][k], out[1][i][k]), k
