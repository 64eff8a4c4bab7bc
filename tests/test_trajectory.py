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


# intervals whose plans have one segment and more, of fewer and of more than
# eight steps (recomputes on one stream and on two), with short first ones
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


# Small domains run the deviation form two steps to a launch, in tiles of 30 x
# 14 cells, and the reference's order in single steps.  In FP64 the two forms round apart by about 1e-14 of the largest
# gradient over these steps; a population taken from a wrong cell is off by
# more than 1e-4 of it.
EDGES = [(1, 1), (2, 3), (13, 29), (14, 30), (15, 31), (28, 60), (29, 61), (1, 95), (43, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("collision", ["BGK", "TRT", "MRT"])
@pytest.mark.parametrize("shape,steps", [(s, n) for s in EDGES for n in (2, 5)])
def test_paired_steps_equal_single_steps(gpu, collision, shape, steps):
    print(f"case pairs {collision} {shape} steps {steps}", flush=True)
    f, a, b = state("D2Q9", shape, "f64", gpu)
    single, pairs = (adjoint.reactive_gradient(collision, f, a, b, steps, 1.6, 1.25, 0.05, 2, fast=fast)
                     for fast in (False, True))
    want = adjoint.loss_of(collision, f, a, b, steps, 1.6, 1.25, 0.05, fast=True)
    assert abs(pairs[0] - want) <= 1e-13 and abs(single[0] - want) <= 1e-13
    for x, y in zip(pairs[1:4], single[1:4]):
        assert (x - y).abs().max().item() <= 1e-11 * y.abs().max().item()
    assert abs(pairs[4] - single[4]) <= 1e-11 * max(abs(single[4]), 1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("fast", [False, True])
def test_paired_gradient_does_not_depend_on_the_segments(gpu, fast):
    print(f"case paired segments fast={fast}", flush=True)
    f, a, b = state("D2Q9", (512, 515), "f32", gpu)
    want, got = (adjoint.reactive_gradient("TRT", f, a, b, 23, 1.6, 1.25, 0.05, iv, fast=fast) for iv in (23, 3))
    assert got[0] == want[0] and got[4] == want[4]
    assert all(torch.equal(x, y) for x, y in zip(got[1:4], want[1:4]))


# From 2^18 cells on the reference's order also runs in pairs; the FP64 sweep of
# an FP32 run steps singly.  Their final states, so their losses, are the same.
@pytest.mark.gpu
@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("collision", ["BGK", "TRT", "MRT"])
def test_paired_loss_equals_single_steps_at_2_18_cells(gpu, collision, fast):
    print(f"case paired loss {collision} fast={fast}", flush=True)
    f, a, b = state("D2Q9", (512, 515), "f32", gpu)
    pairs, single = (adjoint.reactive_gradient(collision, f, a, b, 7, 1.6, 1.25, 0.05, 7, fast=fast, adjoint_f64=w)
                     for w in (False, True))
    assert pairs[0] == single[0]
