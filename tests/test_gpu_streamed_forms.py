"""GPU: the streaming forms of the gradient's kernels and of the 3D steps, which
only domains past the caches on aligned planes take.  A workspace, or a set of
planes, off the cache lines takes the ordinary stores, and tiles another order
of the streaming ones, of the same arithmetic, so the runs must agree bit for
bit.  dloss/d omega_c sums the same cells in another order."""
from __future__ import annotations

import pytest
import torch

import lbcube
from lbcube import adjoint
from lbcube import init as lbinit
from test_trajectory import state

pytestmark = pytest.mark.gpu

# (lattice, shape, storage, FP64 adjoint): two levels of 260 to 300 MiB (the FP64 sweep of an FP32 run 510), planes a
# multiple of 64 bytes
RUNS = [("D2Q9", (1344, 1344), "f32", False), ("D2Q9", (960, 960), "f64", False),
        ("D3Q19", (104, 96, 112), "f32", False), ("D3Q19", (72, 80, 96), "f64", False),
        ("D3Q27", (88, 96, 112), "f32", False), ("D3Q19", (104, 96, 112), "f32", True)]


@pytest.mark.parametrize("collision,fast", [(c, f) for c in ("BGK", "TRT", "MRT") for f in (False, True)] +
                         [("RLBM", False)])
@pytest.mark.parametrize("lattice,shape,storage,wide", RUNS)
def test_streamed_gradient_equals_the_ordinary_one(gpu, lattice, shape, storage, wide, collision, fast):
    print(f"case streamed gradient {lattice} {shape} {collision} {storage} wide={wide} fast={fast}", flush=True)
    f, a, b = state(lattice, shape, storage, gpu)
    assert f[0].numel() * f.element_size() % 64 == 0
    two_levels = 2 * (f.numel() + a.numel() + b.numel()) * f.element_size()
    assert two_levels > 256 << 20
    steps, interval = 7, 2
    nz = shape[0] if len(shape) == 3 else 1
    nbytes = adjoint.workspace_bytes(f.dtype, shape[-1], shape[-2], steps, interval, lbcube.DEFAULT_BLOCK, lattice, nz)
    memory = torch.empty(nbytes + 64, dtype=torch.uint8, device=f.device)
    assert memory.data_ptr() % 64 == 0
    got = []
    for shift in (0, 8):
        got.append(adjoint.reactive_gradient(collision, f, a, b, steps, 1.6, 1.25, 0.05, interval, fast=fast,
                                             adjoint_f64=wide, lattice=lattice,
                                             workspace=memory[shift:shift + nbytes]))
    streamed, ordinary = got
    assert streamed[0] == ordinary[0]
    assert all(torch.equal(x, y) for x, y in zip(streamed[1:4], ordinary[1:4]))
    assert all(bool(torch.isfinite(g).all()) for g in streamed[1:4])
    # FP64 sums over blocks and steps of the same terms: some 30 roundings of the sum of their magnitudes, of which the
    # sum keeps a thousandth or more
    assert abs(streamed[4] - ordinary[4]) <= 1e-11 * abs(ordinary[4])


# 3D steps past the caches against the same in tiles: planes that crowd the cache sets (contiguous blocks), others
# (dispatch order and runs of 8), and planes off the cache lines (ordinary stores)
STEPS_3D = [("D3Q19", (128, 128, 128), "f32"), ("D3Q19", (136, 144, 128), "f32"), ("D3Q19", (112, 112, 112), "f64"),
            ("D3Q19", (144, 136, 160), "f64"), ("D3Q19", (160, 176, 160), "f16"), ("D3Q19", (256, 128, 128), "f16"),
            ("D3Q27", (112, 112, 224), "bf16"), ("D3Q27", (128, 112, 144), "f32"), ("D3Q19", (131, 133, 129), "f32"),
            ("D3Q27", (151, 149, 153), "f16")]


@pytest.mark.parametrize("lattice,shape,storage", STEPS_3D)
def test_3d_reactive_steps_past_the_caches_equal_the_tiled_ones(gpu, lattice, shape, storage):
    print(f"case streamed 3D {lattice} {shape} {storage}", flush=True)
    gen = torch.Generator(device="cpu").manual_seed(3)
    u = (0.02 * torch.randn((3,) + shape, generator=gen, dtype=torch.float32)).double().cuda()
    ca = torch.rand(shape, generator=gen, dtype=torch.float64).cuda()
    ref = 0.5 if storage in ("f16", "bf16") else 0.0
    f = lbinit.equilibrium(lattice, None, u, storage)
    a = lbinit.scalar_equilibrium("D3Q7", ca, u, storage, ref)
    b = lbinit.scalar_equilibrium("D3Q7", 1.0 - ca, u, storage, ref)
    lattices = (lattice, "D3Q7", "D3Q7")
    rows = shape[1]
    tiled = [lbcube.to_tiles(l, t, rows) for l, t in zip(lattices, (f, a, b))]
    new, tnew = [torch.empty_like(t) for t in (f, a, b)], [torch.empty_like(t) for t in tiled]
    fast = storage in ("f16", "bf16")

    def check(what, which):
        for k in which:
            assert torch.equal(lbcube.from_tiles(lattices[k], tnew[k]), new[k]), (what, k)

    lbcube.reactive_fused_step(lattice, "TRT", "D3Q7", f, new[0], a, new[1], b, new[2], 1.6, 1.2, 0.05, ref_a=ref,
                               ref_b=ref, fast=fast)
    lbcube.reactive_fused_step_tiled(lattice, "TRT", "D3Q7", tiled[0], tnew[0], tiled[1], tnew[1], tiled[2], tnew[2],
                                     1.6, 1.2, 0.05, ref_a=ref, ref_b=ref, fast=fast)
    check("fused", (0, 1, 2))
    lbcube.reaction_step(lattice, "D3Q7", a, new[1], b, new[2], f, 1.2, 0.05, ref_a=ref, ref_b=ref)
    lbcube.reaction_step_tiled(lattice, "D3Q7", tiled[1], tnew[1], tiled[2], tnew[2], tiled[0], 1.2, 0.05, ref_a=ref,
                               ref_b=ref)
    check("reaction", (1, 2))
    lbcube.scalar_step(lattice, "D3Q7", a, new[1], f, 1.2, ref=ref)
    lbcube.scalar_step_tiled(lattice, "D3Q7", tiled[1], tnew[1], tiled[0], 1.2, ref=ref)
    check("scalar", (1,))


# Misaligned 2D species steps, which stream where that pays
@pytest.mark.parametrize("shape,storage", [((1501, 1501), "f32"), ((1199, 1201), "f64"), ((2047, 2049), "f32"),
                                           ((1499, 1501), "f64"), ((1949, 1951), "f32"), ((2501, 2500), "f16")])
def test_misaligned_2d_species_steps_equal_the_tiled_ones(gpu, shape, storage):
    print(f"case misaligned species {shape} {storage}", flush=True)
    gen = torch.Generator(device="cpu").manual_seed(3)
    u = (0.02 * torch.randn((2,) + shape, generator=gen, dtype=torch.float32)).double().cuda()
    ca = torch.rand(shape, generator=gen, dtype=torch.float64).cuda()
    ref = 0.5 if storage == "f16" else 0.0
    f = lbinit.equilibrium("D2Q9", None, u, storage)
    a = lbinit.scalar_equilibrium("D2Q5", ca, u, storage, ref)
    b = lbinit.scalar_equilibrium("D2Q5", 1.0 - ca, u, storage, ref)
    tiled = [lbcube.to_tiles(l, t, 1) for l, t in (("D2Q9", f), ("D2Q5", a), ("D2Q5", b))]
    new, tnew = [torch.empty_like(t) for t in (a, b)], [torch.empty_like(t) for t in tiled[1:]]
    lbcube.reaction_step("D2Q9", "D2Q5", a, new[0], b, new[1], f, 1.2, 0.05, ref_a=ref, ref_b=ref)
    lbcube.reaction_step_tiled("D2Q9", "D2Q5", tiled[1], tnew[0], tiled[2], tnew[1], tiled[0], 1.2, 0.05, ref_a=ref,
                               ref_b=ref)
    assert torch.equal(lbcube.from_tiles("D2Q5", tnew[0]), new[0])
    assert torch.equal(lbcube.from_tiles("D2Q5", tnew[1]), new[1])
    lbcube.scalar_step("D2Q9", "D2Q5", a, new[0], f, 1.2, ref=ref)
    lbcube.scalar_step_tiled("D2Q9", "D2Q5", tiled[1], tnew[0], tiled[0], 1.2, ref=ref)
    assert torch.equal(lbcube.from_tiles("D2Q5", tnew[0]), new[0])
