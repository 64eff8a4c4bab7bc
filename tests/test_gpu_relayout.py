"""GPU: layout conversions (lbc_relayout, lbc_relayout_tiled) at every width of
the vectors they move: runs, strides or addresses that are multiples of 16, 8,
4 or 2 bytes only, and counts around the vectors of one block, against torch's
permutation of the axes."""
from __future__ import annotations

import pytest
import torch

import lbcube

pytestmark = pytest.mark.gpu

DTYPES = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def pattern(shape, dtype):
    n = 1
    for v in shape:
        n *= v
    v = torch.arange(n, dtype=torch.int64, device="cuda") * 40503 % 65521
    bits = {2: torch.int16, 4: torch.int32, 8: torch.int64}[torch.empty(0, dtype=dtype).element_size()]
    return v.to(bits).view(dtype).view(shape)


def same(a, b):
    return torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


# one element, odd runs, and runs of 4096 +- a vector: whole, one over and one short of a block's vectors
@pytest.mark.parametrize("nx,ny,nz", [(1, 1, 1), (5, 7, 3), (6, 5, 4), (12, 5, 3), (8, 8, 8), (64, 64, 2), (64, 65, 2),
                                      (129, 63, 5), (128, 33, 7)])
@pytest.mark.parametrize("storage", list(DTYPES))
def test_slabs_and_tiles_both_ways(gpu, storage, nx, ny, nz):
    print(f"case relayout {storage} {nx} x {ny} x {nz}", flush=True)
    f = pattern((19, nz, ny, nx), DTYPES[storage])
    h = lbcube.to_slabs("D3Q19", f)
    assert same(h, f.permute(1, 0, 2, 3))
    assert same(lbcube.from_slabs("D3Q19", h), f)
    for rows in sorted({1, ny} | {r for r in (5, 7, 13) if ny % r == 0}):
        g = f[:9, 0].contiguous()
        t = lbcube.to_tiles("D2Q9", g, rows)
        assert same(t, g.view(9, ny // rows, rows, nx).permute(1, 0, 2, 3)), rows
        assert same(lbcube.from_tiles("D2Q9", t), g), rows


@pytest.mark.parametrize("storage", list(DTYPES))
def test_addresses_and_strides_off_the_vector_boundaries(gpu, storage):
    nx, ny, nz, q = 32, 16, 5, 19
    dtype = DTYPES[storage]
    f = pattern((q, nz, ny, nx), dtype)
    want = f.permute(1, 0, 2, 3).contiguous()
    for shift in (0, 1, 2, 4):
        src = torch.zeros(f.numel() + 8, dtype=dtype, device="cuda")[shift:shift + f.numel()]
        src.copy_(f.view(-1))
        for pad in (0, 1, 2, 8):
            plane = nx * ny + pad
            slab = q * plane + pad
            dst = torch.zeros(nz * slab + 8, dtype=dtype, device="cuda")[shift:]
            lbcube.relayout("D3Q19", src, dst, (nx, ny, nz), (0, 0), (plane, slab))
            got = dst[:nz * slab].view(nz, slab)
            planes = got[:, :q * plane].reshape(nz, q, plane)
            assert same(planes[:, :, :nx * ny].reshape(nz, q, ny, nx), want), (shift, pad)
            assert not torch.any(planes[:, :, nx * ny:].contiguous().view(torch.uint8)), (shift, pad)
            back = torch.zeros_like(src)
            lbcube.relayout("D3Q19", dst, back, (nx, ny, nz), (plane, slab), (0, 0))
            assert same(back, src), (shift, pad)
