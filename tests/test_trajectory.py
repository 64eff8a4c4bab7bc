"""The gradient's trajectory: the plan that cuts a run into segments (the
header's own code on the host), and gradients that do not depend on it.  A
recomputed segment and a kept one hold the same values, so runs of one, two and
many segments, on one stream or two, agree bit for bit."""
from __future__ import annotations

import os
import subprocess

import pytest
import torch

from lbcube import adjoint
from lbcube import init as lbinit

HERE = os.path.dirname(os.path.abspath(__file__))


def test_plan_fits_and_covers(tmp_path):
    exe = tmp_path / "trajectory_check"
    subprocess.run(["g++", "-O2", "-std=c++20", os.path.join(HERE, "trajectory_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "ok 252000\n", r.stdout + r.stderr


def state(lattice, shape, dtype, gpu):
    g = torch.Generator(device="cpu").manual_seed(5)
    u = 0.02 * torch.randn((len(shape),) + shape, generator=g, dtype=torch.float64).to(gpu)
    c = torch.rand(shape, generator=g, dtype=torch.float64).to(gpu)
    species = adjoint.SPECIES[lattice]
    return (lbinit.equilibrium(lattice, None, u, dtype), lbinit.scalar_equilibrium(species, c, u, dtype),
            lbinit.scalar_equilibrium(species, 1.0 - c, u, dtype))


# intervals whose plans have one segment, two, and more of fewer and of more
# than eight steps (recomputes on one stream and on two), with short first ones
CASES = [("D2Q9", (13, 37), "MRT", "f32", False, (1, 4, 5, 7)), ("D2Q9", (32, 64), "TRT", "f64", False, (1, 5, 6)),
         ("D3Q19", (5, 9, 11), "TRT", "f32", False, (1, 3, 4, 6)), ("D3Q19", (8, 8, 16), "MRT", "f64", False, (2, 5)),
         ("D3Q27", (6, 7, 9), "BGK", "f32", False, (2, 5)), ("D3Q27", (6, 7, 9), "MRT", "f32", False, (2, 5)),
         ("D2Q9", (13, 37), "RLBM", "f32", False, (1, 4, 9)), ("D3Q19", (5, 9, 11), "BGK", "f32", True, (1, 4, 9))]


@pytest.mark.gpu
@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("lattice,shape,collision,storage,wide,intervals", CASES)
def test_gradient_does_not_depend_on_the_segments(gpu, lattice, shape, collision, storage, wide, intervals, fast):
    print(f"case trajectory {lattice} {shape} {collision} {storage} wide={wide} fast={fast}", flush=True)
    f, a, b = state(lattice, shape, storage, gpu)
    steps = 40
    keep = [t.clone() for t in (f, a, b)]
    run = lambda interval: adjoint.reactive_gradient(collision, f, a, b, steps, 1.6, 1.25, 0.05, interval,  # noqa: E731
                                                     fast=fast, adjoint_f64=wide, lattice=lattice)
    want = run(steps)
    assert all(bool(torch.isfinite(g).all()) for g in want[1:4])
    for interval in intervals:
        got = run(interval)
        assert got[0] == want[0] and got[4] == want[4], interval
        assert all(torch.equal(x, y) for x, y in zip(got[1:4], want[1:4])), interval
    assert all(torch.equal(x, y) for x, y in zip((f, a, b), keep))
