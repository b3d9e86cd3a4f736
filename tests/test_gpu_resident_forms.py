"""The resident loop on random forms of what it accepts: grids of every aspect (a column or a row of
tiles, strips), CPML of any width or none, both orders, the free surface, the three types, sources
and receivers anywhere (frame cells and corners, several in one cell, none), uneven records, windows
with strides, every store and the exact gradient; against the split step, bit for bit."""
import random

import numpy as np
import pytest

import psv_oracle as O
import refcase as RC
from gpucase import plan_of
from test_gpu_parity import MEMS
from test_gpu_resident import _same

pytestmark = pytest.mark.gpu


def _size(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(max(lo + 1, hi))))))


def _draw(rng):
    order, npml, prec = rng.choice([2, 4]), rng.choice([0, 1, 2, 5, 8, 20]), rng.choice(["fp32", "fp32", "fp64", "fp32x2"])
    lo = max(16, 2 * npml + order + 3)
    form = rng.choice(["row", "column", "any", "any", "any", "strips"])
    nxt, nzt = _size(rng, lo, 1200), _size(rng, lo, 600)
    if form == "row":
        nxt, nzt = _size(rng, lo, 3000), lo + rng.randint(0, 3)
    elif form == "column":
        nxt, nzt = lo + rng.randint(0, 3), _size(rng, lo, 3000)
    elif form == "strips" and prec != "fp32x2":
        nxt, nzt = (_size(rng, 1500, 2600), _size(rng, 700, 1000)) if prec == "fp32" else (_size(rng, 900, 1400), _size(rng, 600, 800))
    elif prec != "fp32":
        nzt = max(lo, min(nzt, 300000 // nxt))
    return dict(order=order, fsurf=rng.randint(0, 1), npml=npml, prec=prec, nxt=nxt, nzt=nzt, nt=rng.choice([17, 40, 66]),
                shots=rng.choice([1, 1, 2, 3, 5]), kmax=rng.choice([1.0, 1.7]), k=rng.choice([8, 11, 30]),
                mode=rng.choice(["full", "full", "checkpoint", "discrete", "discrete"]), energy=rng.random() < 0.5)


def _points(rng, c, count, comps):
    H, nxt, nzt = c["order"] // 2, c["nxt"], c["nzt"]
    p = [(rng.choice([0, 1, H, nxt - 1, nxt - H - 1, rng.randrange(nxt), rng.randrange(nxt)]),
          rng.choice([0, H, H + 1, nzt - 1, rng.randrange(nzt), rng.randrange(nzt)]), rng.choice(comps)) for _ in range(count)]
    p += p[:rng.randint(0, len(p))]
    return dict(zip(("x", "z", "comp"), map(list, zip(*p)))) if p else dict(x=[], z=[], comp=[])


@pytest.mark.parametrize("seed", range(48))
def test_form(seed):
    rng = random.Random(seed)
    c = _draw(rng)
    print(f"form {seed} {c}", flush=True)
    H = c["order"] // 2
    ppad = c["npml"] + H
    pb = RC.small_problem(nx=c["nxt"] - 2 * ppad, nz=c["nzt"] - (ppad + H if c["fsurf"] else 2 * ppad), npml=c["npml"],
                          nt=c["nt"], fsurf=c["fsurf"], fdorder=c["order"], seed=seed, hetero=c["nxt"] * c["nzt"] < 200000)
    assert (pb.nxt, pb.nzt) == (c["nxt"], c["nzt"])
    pb.pml = O.cpml_pro(c["npml"], 5.0, 25.0, 2.0, c["kmax"], 1e-3, 2750.0, 5e-4)
    x1, z1 = rng.randint(0, pb.nxt // 2), rng.randint(0, pb.nzt // 2)
    pb.fwi = dict(dt=rng.choice([1, 2, 5]), dx=rng.choice([1, 1, 2, 3]), dz=rng.choice([1, 1, 2, 7]),
                  x1=x1, x2=rng.randint(x1, pb.nxt), z1=z1, z2=rng.randint(z1, pb.nzt))
    comps = [1, 2] if c["mode"] == "discrete" else [1, 2, 4]
    shots, obs = [], []
    for s in range(c["shots"]):
        nt = c["nt"] if s == 0 else rng.randint(1, c["nt"])
        src, rec = _points(rng, c, rng.choice([0, 1, 6]) if s else 3, comps), _points(rng, c, rng.choice([0, 1, 40]) if s else 9, [1, 2])
        noise = np.random.default_rng([seed, s])
        shots.append(dict(nt=nt, src=src, rec=rec,
                          src_signal=noise.standard_normal((len(src["x"]), nt)) * np.hanning(nt + 2)[1:-1]))
        obs.append(1e-3 * noise.standard_normal((len(rec["x"]), nt)))
    out = []
    for tz in (8, None):
        plan = plan_of(pb, c["prec"], tz=tz, shots=shots)
        if c["mode"] == "discrete":
            plan.set_gradient_mode("discrete", c["k"])
        else:
            plan.set_store_mode(c["mode"], c["k"])
        names = ["vx", "vz", "sxx", "szx", "szz", "We"] + list(MEMS if c["npml"] else ())
        fields = lambda names: [plan.field(a, s) for a in names for s in range(c["shots"])]
        plan.forward(energy=c["energy"], gradient=True)
        r = [plan.records(s) for s in range(c["shots"])] + fields(names) + [plan.misfit(obs)]
        plan.adjoint(energy=c["energy"], gradient=True)
        for s in range(-1, c["shots"]):
            r += (list(plan.coefficient_gradient(s).values()) + list(plan.model_gradient(s)) if c["mode"] == "discrete"
                  else list(plan.gradient(s)))
        if c["mode"] != "discrete":
            r += fields(names + ["ux", "uz"])
        plan.close()
        out.append(r)
    assert all(np.isfinite(a).all() for a in out[0])
    assert all(_same(a, b) for a, b in zip(*out)), [k for k, (a, b) in enumerate(zip(*out)) if not _same(a, b)]
