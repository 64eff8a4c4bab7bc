"""The gradient's schedule as the library plans it (the header's own code,
compiled on the host), for tests that have to reach a certain one."""
from __future__ import annotations

import collections
import functools
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
LATTICE = {"D2Q9": (2, 9, 5), "D3Q19": (3, 19, 7), "D3Q27": (3, 27, 7)}
PAIR_CELLS = 1 << 18  # the reference's order runs in pairs from here on
Schedule = collections.namedtuple("Schedule", "length segments first overlapped")


@functools.lru_cache(maxsize=None)
def _checker():
    folder = tempfile.TemporaryDirectory()
    exe = os.path.join(folder.name, "schedule_check")
    subprocess.run(["g++", "-O2", "-std=c++20", os.path.join(HERE, "schedule_check.cpp"), "-o", exe], check=True,
                   capture_output=True, timeout=300)
    return exe, folder


def schedule(lattice, shape, collision, storage, steps, interval, fast=False, wide=False):
    """The schedule of reactive_gradient for these arguments (wide: the FP64
    adjoint of an FP32 run)."""
    dim, qf, qs = LATTICE[lattice]
    cells = 1
    for n in shape:
        cells *= n
    compact = collision != "RLBM" and not wide
    element = 8 if storage == "f64" else 4
    paired = compact and dim == 2 and (fast or cells >= PAIR_CELLS)
    line = f"{dim} {qf} {qs} {int(compact)} {steps} {interval} {cells} {element} {int(paired)}\n"
    r = subprocess.run([_checker()[0]], input=line, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    length, segments, first, over = (int(v) for v in r.stdout.split())
    return Schedule(length, segments, first, bool(over))
