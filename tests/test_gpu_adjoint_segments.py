"""GPU: the discrete adjoint against the oracle's FP64 CPU adjoint on runs that
the library does cut: three segments or more, so that checkpoints, the recompute
of a segment and, from segments of eight steps on, the second stream are on the
way.  The schedule is the library's own (schedules.py) and asserted."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import test_oracle_adjoint as TA
import test_oracle_adjoint_3d as TA3
from lbcube import adjoint as ADJ
from oracle import oracle as O
from schedules import schedule

STEPS = 40
# fluid lattice, extents (x first), blocks: small and larger than one block, the default and the 1024-work-item kernels
DOMAINS = [("D2Q9", (12, 10), (None, (1024, 1, 1))), ("D2Q9", (60, 50), (None, (32, 32, 1))),
           ("D3Q19", (7, 6, 5), (None, (1024, 1, 1))), ("D3Q19", (12, 10, 9), (None, (16, 16, 4))),
           ("D3Q27", (7, 6, 5), (None, (16, 16, 4)))]


def interval_of(collision):
    return 8 if collision == "RLBM" else 4


def planned(lattice, extents, collision, fast=False):
    return schedule(lattice, extents, collision, "f64", STEPS, interval_of(collision), fast)


def test_the_runs_are_cut():
    both = set()
    for lattice, extents, _ in DOMAINS:
        for collision in ("BGK", "TRT", "MRT", "RLBM"):
            s = planned(lattice, extents, collision)
            assert s.segments >= 3, (lattice, extents, collision, s)
            both.add(s.overlapped)
    assert both == {False, True}


def state(lattice, extents):
    if lattice == "D2Q9":
        return TA.small_state(nx=extents[0], ny=extents[1], seed=4)
    return TA3.small_state_3d(lattice, nx=extents[0], ny=extents[1], nz=extents[2], seed=4)


def dev(x, gpu):
    return torch.from_numpy(np.ascontiguousarray(x)).to(gpu).to(torch.float64)


# The 17-step bounds of test_gpu_adjoint.py times 40 / 17, rounded up: the
# rounding of a step is passed on by the linear sweep, which does not amplify it.
@pytest.mark.gpu
@pytest.mark.parametrize("collision", ["BGK", "TRT", "MRT", "RLBM"])
@pytest.mark.parametrize("lattice,extents,blocks", DOMAINS)
def test_cut_runs_match_the_oracle(gpu, lattice, extents, blocks, collision):
    f, a, b = state(lattice, extents)
    omega, omega_c, k = 1 / 0.7, 1 / 0.9, 0.4
    kw = {} if lattice == "D2Q9" else {"lattice": lattice}
    J, gf, ga, gb, dw = O.reactive_gradient(collision, "f64", f, a, b, omega, omega_c, k, STEPS, **kw)
    for block in blocks:
        print(f"case cut adjoint {lattice} {extents} {collision} block={block}", flush=True)
        got = ADJ.reactive_gradient(collision, dev(f, gpu), dev(a, gpu), dev(b, gpu), STEPS, omega, omega_c, k,
                                    interval=interval_of(collision), block=block, **kw)
        assert abs(got[0] - J) <= 3e-13 * abs(J)
        for g, want in zip(got[1:4], (gf, ga, gb)):
            assert np.max(np.abs(g.cpu().numpy() - want)) <= 3e-12 * np.max(np.abs(want))
        assert abs(got[4] - dw) <= 3e-11 * abs(dw)


# The deviation form rounds apart from the reference's order (test_gpu_adjoint.py's bounds).
@pytest.mark.gpu
@pytest.mark.parametrize("collision", ["BGK", "TRT", "MRT"])
@pytest.mark.parametrize("lattice,extents,blocks", DOMAINS)
def test_cut_runs_of_the_deviation_form_match_the_oracle(gpu, lattice, extents, blocks, collision):
    assert planned(lattice, extents, collision, True).overlapped
    f, a, b = state(lattice, extents)
    omega, omega_c, k = 1 / 0.6, 1 / 0.8, 0.2
    kw = {} if lattice == "D2Q9" else {"lattice": lattice}
    J, gf, ga, gb, dw = O.reactive_gradient(collision, "f64", f, a, b, omega, omega_c, k, STEPS, **kw)
    for block in blocks:
        print(f"case cut adjoint, deviation form, {lattice} {extents} {collision} block={block}", flush=True)
        got = ADJ.reactive_gradient(collision, dev(f, gpu), dev(a, gpu), dev(b, gpu), STEPS, omega, omega_c, k,
                                    interval=interval_of(collision), block=block, fast=True, **kw)
        assert abs(got[0] - J) <= 1e-12 * abs(J) and abs(got[4] - dw) <= 1e-9 * abs(dw)
        for g, want in zip(got[1:4], (gf, ga, gb)):
            assert np.max(np.abs(g.cpu().numpy() - want)) <= 1e-9 * np.max(np.abs(want))
