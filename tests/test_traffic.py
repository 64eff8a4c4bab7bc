"""Store form and block order of the steps (plan_traffic and block_at of
lb-cube_amd/csrc/lbc_launch.hpp): the block renumbering is a bijection of every
grid (the header's own code on the host), and a step's values do not depend on
the form it takes.  Domains just above the cache limit on aligned planes
stream their stores; planes one element further apart, or tiles, take another
form or order of the same step, so the two runs must agree bit for bit."""
from __future__ import annotations

import os
import subprocess

import pytest
import torch

import lbcube
from lbcube import init as lbinit

HERE = os.path.dirname(os.path.abspath(__file__))


def test_block_order_is_a_bijection(tmp_path):
    exe = tmp_path / "block_order_check"
    subprocess.run(["/opt/rocm/bin/hipcc", "-O2", "-std=c++23", "--offload-arch=gfx950", "-x", "hip",
                    os.path.join(HERE, "block_order_check.cpp"), "-o", str(exe)], check=True, capture_output=True,
                   timeout=300)
    sizes = list(range(1, 70)) + [255, 256, 257, 511, 512, 513, 1023, 2048, 16384, 31524, 65537]
    cases = [(n, o) for n in sizes for o in (0, 1, 3, 5, 31)]
    r = subprocess.run([str(exe)], input="".join(f"{n} {o}\n" for n, o in cases), capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0 and r.stdout == f"ok {len(cases)}\n", r.stdout + r.stderr


def velocity(shape):
    g = torch.Generator(device="cpu").manual_seed(3)
    u = 0.02 * torch.randn((len(shape),) + tuple(shape), generator=g, dtype=torch.float32)
    return u.double().cuda()


# (lattice, extents, storage): two levels of 371 to 400 MB, just above the
# limit, planes and rows on multiples of 64 bytes
STREAMED = [("D2Q9", (1664, 1552), "f64"), ("D2Q9", (2368, 2176), "f32"), ("D2Q9", (3328, 3136), "f16"),
            ("D3Q19", (112, 104, 112), "f64"), ("D3Q19", (144, 132, 130), "f32"), ("D3Q19", (160, 176, 176), "f16"),
            ("D3Q27", (160, 160, 136), "bf16")]


@pytest.mark.gpu
@pytest.mark.parametrize("lattice,extents,storage", STREAMED)
def test_streamed_step_equals_the_step_on_spaced_planes(gpu, lattice, extents, storage):
    print(f"case streamed {lattice} {extents} {storage}", flush=True)
    shape = extents[::-1]
    f = lbinit.equilibrium(lattice, None, velocity(shape), storage)
    q, cells = f.shape[0], f[0].numel()
    got = torch.empty_like(f)
    lbcube.fluid_step(lattice, "TRT", f, got, 1.6, fast=True)
    pitch = cells + 1  # every plane on another offset from the cache lines
    spaced = torch.zeros(q * pitch, dtype=f.dtype, device=f.device)
    out = torch.zeros_like(spaced)
    spaced.view(q, pitch)[:, :cells] = f.view(q, cells)
    lbcube.fluid_step_pitched(lattice, "TRT", spaced, out, extents + ((1,) if len(extents) == 2 else ()), pitch, 1.6,
                              fast=True)
    assert torch.equal(out.view(q, pitch)[:, :cells], got.view(q, cells))
    assert not torch.any(out.view(q, pitch)[:, cells:])


@pytest.mark.gpu
@pytest.mark.parametrize("storage,nx,ny", [("f64", 1184, 1040), ("f32", 1664, 1504), ("f16", 2400, 2080)])
def test_streamed_reactive_steps_equal_the_tiled_ones(gpu, storage, nx, ny):
    print(f"case streamed reactive {storage} {nx} x {ny}", flush=True)
    u = velocity((ny, nx))
    ref = 0.5 if storage == "f16" else 0.0
    f = lbinit.equilibrium("D2Q9", None, u, storage)
    ca = torch.rand((ny, nx), dtype=torch.float64, device="cuda")
    a = lbinit.scalar_equilibrium("D2Q5", ca, u, storage, ref)
    b = lbinit.scalar_equilibrium("D2Q5", 1.0 - ca, u, storage, ref)
    tf, ta, tb = (lbcube.to_tiles(l, t, 16) for l, t in (("D2Q9", f), ("D2Q5", a), ("D2Q5", b)))
    new, tnew = [torch.empty_like(t) for t in (f, a, b)], [torch.empty_like(t) for t in (tf, ta, tb)]

    def check(names):
        for k, name in names:
            lat = "D2Q9" if k == 0 else "D2Q5"
            assert torch.equal(lbcube.from_tiles(lat, tnew[k]), new[k]), name

    lbcube.reactive_fused_step("D2Q9", "TRT", "D2Q5", f, new[0], a, new[1], b, new[2], 1.6, 1.2, 0.05, ref_a=ref,
                               ref_b=ref)
    lbcube.reactive_fused_step_tiled("D2Q9", "TRT", "D2Q5", tf, tnew[0], ta, tnew[1], tb, tnew[2], 1.6, 1.2, 0.05,
                                     ref_a=ref, ref_b=ref)
    check([(0, "fluid"), (1, "A"), (2, "B")])
    lbcube.reaction_step("D2Q9", "D2Q5", a, new[1], b, new[2], f, 1.2, 0.05, ref_a=ref, ref_b=ref)
    lbcube.reaction_step_tiled("D2Q9", "D2Q5", ta, tnew[1], tb, tnew[2], tf, 1.2, 0.05, ref_a=ref, ref_b=ref)
    check([(1, "A of the reaction step"), (2, "B of the reaction step")])
    lbcube.scalar_step("D2Q9", "D2Q5", a, new[1], f, 1.2, ref=ref)
    lbcube.scalar_step_tiled("D2Q9", "D2Q5", ta, tnew[1], tf, 1.2, ref=ref)
    check([(1, "the passive scalar")])
