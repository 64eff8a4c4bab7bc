"""When the gradient recomputes its segments on a second stream (the rule of
lbc_trajectory.hpp, on the host), and that this schedule leaves the gradient as
it is, bit for bit, on the default stream and on a caller's."""
from __future__ import annotations

import pytest
import torch

from lbcube import adjoint
from schedules import schedule
from test_trajectory import state

# (lattice, shape, collision, storage, fast, FP64 adjoint, steps, interval), each recomputed on the second stream in
# at least three segments: single steps and pairs (the deviation form, and from 2^18 cells the reference's order), every
# kind of trajectory, states from 0.04 to 20 MiB
OVERLAPPED = [("D2Q9", (190, 200), "BGK", "f64", False, False, 40, 4),
              ("D2Q9", (190, 200), "TRT", "f64", True, False, 40, 4),
              ("D2Q9", (310, 300), "MRT", "f32", False, False, 41, 4),
              ("D2Q9", (48, 64), "BGK", "f32", False, False, 200, 32),
              ("D2Q9", (13, 37), "MRT", "f32", True, False, 40, 4),
              ("D2Q9", (512, 515), "TRT", "f32", False, False, 27, 5),
              ("D2Q9", (512, 515), "BGK", "f32", True, False, 28, 5),
              ("D2Q9", (90, 100), "RLBM", "f64", False, False, 50, 8),
              ("D2Q9", (200, 300), "BGK", "f32", True, True, 50, 8),
              ("D3Q19", (12, 10, 11), "TRT", "f32", True, False, 60, 5),
              ("D3Q19", (20, 24, 16), "MRT", "f64", False, False, 40, 4),
              ("D3Q27", (9, 8, 10), "BGK", "f64", False, False, 60, 5),
              ("D3Q19", (12, 10, 11), "RLBM", "f32", False, False, 50, 8),
              ("D3Q19", (12, 10, 11), "BGK", "f32", False, True, 50, 8)]


def test_states_that_leave_the_gpu_idle_are_overlapped():
    for case in OVERLAPPED:
        lattice, shape, collision, storage, fast, wide, steps, interval = case
        s = schedule(lattice, shape, collision, storage, steps, interval, fast, wide)
        assert s.overlapped and s.segments > 2 and s.length >= 8, (case, s)
        assert not schedule(lattice, shape, collision, storage, steps, steps, fast, wide).overlapped
    # RLBM and 3D states of any size below the limit
    for n in (64, 96, 128, 256):
        assert schedule("D2Q9", (n, n), "RLBM", "f64", 1024, 32).overlapped, n
    for n in (8, 12, 16, 24, 32, 48):
        for storage in ("f32", "f64"):
            assert schedule("D3Q19", (n, n, n), "RLBM", storage, 300, 16).overlapped, (n, storage)
            assert schedule("D3Q19", (n, n, n), "TRT", storage, 300, 16, True).overlapped, (n, storage)
    # short segments of steps shorter than a launch, large states and few segments are not
    assert not schedule("D2Q9", (128, 128), "RLBM", "f32", 400, 16).overlapped
    assert schedule("D2Q9", (240, 240), "RLBM", "f32", 400, 16).overlapped
    assert schedule("D2Q9", (128, 128), "RLBM", "f32", 1024, 32).overlapped
    assert not schedule("D2Q9", (32, 32), "TRT", "f64", 400, 16).overlapped
    assert schedule("D2Q9", (48, 48), "TRT", "f64", 400, 16).overlapped
    assert not schedule("D2Q9", (1024, 1024), "BGK", "f32", 256, 16, True).overlapped
    assert not schedule("D2Q9", (200, 200), "BGK", "f32", 23, 3, True).overlapped
    assert not schedule("D2Q9", (200, 200), "BGK", "f32", 40, 40, True).overlapped


@pytest.mark.gpu
@pytest.mark.parametrize("lattice,shape,collision,storage,fast,wide,steps,interval", OVERLAPPED)
def test_overlapped_gradient_equals_one_segment(gpu, lattice, shape, collision, storage, fast, wide, steps, interval):
    print(f"case overlapped {lattice} {shape} {collision} {storage} fast={fast} wide={wide}", flush=True)
    f, a, b = state(lattice, shape, storage, gpu)
    run = lambda iv: adjoint.reactive_gradient(collision, f, a, b, steps, 1.6, 1.25, 0.05, iv, fast=fast,  # noqa: E731
                                               adjoint_f64=wide, lattice=lattice)
    want = run(steps)
    assert all(bool(torch.isfinite(g).all()) for g in want[1:4])
    got = [run(interval)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got.append(run(interval))
    torch.cuda.synchronize()
    for g in got:
        assert g[0] == want[0] and g[4] == want[4]
        assert all(torch.equal(x, y) for x, y in zip(g[1:4], want[1:4]))
