// Launch validation shared by every C entry point.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>

#include "lbc_lattice.hpp"
#include "lbc_storage.hpp"

namespace lbc {

inline bool is_2d(int lattice) { return lattice == kD2Q9 || lattice == kD2Q5; }

// Populations per cell of a lattice code (0: unknown).
inline int q_of(int lattice) {
    switch (lattice) {
        case kD2Q9: return 9;
        case kD3Q19: return 19;
        case kD3Q27: return 27;
        case kD2Q5: return 5;
        case kD3Q7: return 7;
        default: return 0;
    }
}

// Division by a launch constant d (1 <= d < 2^32) of any dividend n < 2^32,
// with the add-back form of Granlund & Montgomery's round-up reciprocal
// (PLDI 1994, Fig. 4.1): l = ceil(log2 d), m = floor(2^32 (2^l - d) / d) + 1
// (< 2^32), t = hi32(m n), q = (t + ((n - t) >> min(l, 1))) >> max(l - 1, 0).
// The 33-bit multiplier 2^32 + m exceeds 2^(32+l) / d by at most one unit, so
// n (2^32 + m) / 2^(32+l) exceeds n / d by less than 2^-l <= 1/d and its floor
// is the quotient; the add-back evaluates floor((n + t) / 2^l) without a
// 33-bit intermediate.
struct FastDiv {
    uint32_t m, s1, s2;
};

inline FastDiv make_fastdiv(uint32_t d) {
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    const uint64_t m = ((((1ull << l) - d) << 32) / d) + 1;
    return FastDiv{static_cast<uint32_t>(m), l < 1 ? l : 1u, l > 1 ? l - 1 : 0u};
}

__host__ __device__ __forceinline__ uint32_t fast_div(uint32_t n, FastDiv f) {
    const uint32_t t = static_cast<uint32_t>((static_cast<uint64_t>(n) * f.m) >> 32);  // v_mul_hi_u32
    return (t + ((n - t) >> f.s1)) >> f.s2;
}

// Cells of a domain numbered linearly, x fastest ((z * ny + y) * nx + x): the
// kernels map work-item p of the launch to cell p, so every wave covers 64
// consecutive cells whatever nx and the block shape are (no idle lanes at row
// ends beyond the last wave of the domain).
// Tiles.  A population buffer may be stored in tiles of `rows` rows (rows
// divides ny; rows = ny makes each xy-slab one tile), `tiles` = ny / rows of
// them per xy-slab.  zgap: elements between the end of one tile of a population
// plane and the start of the next (0 in the reference's [Q][Z][Y][X] planes;
// (Q - 1) x the tile's cells when each tile holds its Q planes back to back,
// e.g. the slab order [Z][Q][Y][X]).  Cell (x, y, z) of tile
// t = (z ny + y) / rows lies at element (z ny + y) nx + x + t zgap of its
// population plane.  Without tiles rows = ny and tiles = 1.
struct Cells {
    uint32_t nx, ny, nz, count;
    FastDiv by_nx, by_ny;
    uint32_t zgap;
    uint32_t rows, tiles;
    FastDiv by_rows;
    uint32_t order;  // of the blocks: ordered_block
};

struct CellCoord {
    int x, y, z;
};

// Block orders (ordered_block, below).
constexpr uint32_t kXcds = 8;
constexpr uint32_t kDispatchOrder = 0, kContiguousOrder = 31;

__device__ __forceinline__ CellCoord cell_coord(uint32_t p, const Cells& c) {
    const uint32_t row = fast_div(p, c.by_nx);
    const uint32_t z = fast_div(row, c.by_ny);
    return CellCoord{static_cast<int>(p - row * c.nx), static_cast<int>(row - z * c.ny), static_cast<int>(z)};
}

// The pull sources of destination cell p at coordinates q, for planes whose
// tiles are spaced `zgap` elements apart (Cells); pull.dst is the cell's
// element offset within its plane.  A z step moves nx ny + tiles zgap; a y
// step that crosses a tile boundary moves zgap further (the wrap from the
// last row of a slab to its first crosses tiles - 1 of them).  zgap = 0 and
// one tile per slab give the reference's offsets; the y-tile arithmetic runs
// only when a slab holds several tiles (a wave-uniform branch).
template <int D>
__device__ __forceinline__ Pull locate(uint32_t p, const CellCoord& q, const Cells& c, uint32_t zgap) {
    const uint32_t slab_gap = c.tiles * zgap;  // the gaps of one xy-slab's tiles
    Pull pull(p + static_cast<uint32_t>(q.z) * slab_gap, q.x, q.y, q.z, static_cast<int>(c.nx),
              static_cast<int>(c.ny), static_cast<int>(c.nz), slab_gap);
    if (c.tiles > 1) {
        const uint32_t y = static_cast<uint32_t>(q.y);
        const uint32_t t = fast_div(y, c.by_rows);
        const uint32_t r = y - t * c.rows;
        const uint32_t row = c.nx;
        const uint32_t last = (c.tiles - 1u) * zgap + row * (c.ny - 1u);  // row 0 -> row ny - 1
        pull.dst += t * zgap;
        pull.ym = y == 0 ? last : (r == 0 ? 0u - row - zgap : 0u - row);
        pull.yp = y + 1 == c.ny ? 0u - last : (r + 1 == c.rows ? row + zgap : row);
    }
    return pull;
}

struct LaunchShape {
    dim3 grid, block;  // 1D: ceil(cells / threads) blocks of `threads` work-items
    int nx, ny, nz;
    Cells cells;
    unsigned threads() const { return block.x; }
};

// Kernels are compiled twice, for blocks of up to 256 work-items (the
// register budget the library tunes for) and up to 1024 (the largest block
// HIP accepts, which the reference's launcher also accepts).  The block shape
// the caller passes sets the work-items per block (bx * by * bz); the cells
// are covered linearly.

// Largest domain: 2^32 - 2^20 cells (4,293,918,720), e.g. 1,600^3; 1,200^3
// D3Q19 populations in FP32 ping-pong take 245 GiB of HBM.
constexpr uint64_t kMaxCells = (1ull << 32) - (1ull << 20);
// Coordinates are int.
constexpr uint64_t kMaxExtent = (1ull << 31) - 1;
// HIP's limit on blocks per launch along x.
constexpr uint64_t kMaxBlocks = (1ull << 31) - 1;

// Elements a lane's offset spans within a population plane: the cell count,
// or more when the slabs are spaced apart (zgap).
inline uint64_t lane_extent(const Cells& c) {
    return static_cast<uint64_t>(c.count) + (static_cast<uint64_t>(c.nz) * c.tiles - 1) * c.zgap;
}

// Population planes of more than 4 GiB take 64-bit per-lane addresses (the
// kernels' WIDE instantiation); smaller planes keep the 32-bit byte offsets.
template <class S> bool wide_planes(const LaunchShape& s) {
    return lane_extent(s.cells) * sizeof(S) > (1ull << 32);
}

// Validation order of src/lattice_cuda.cu:488-503: pointers, block, 2D
// normalisation, extents.  Then this library's own limits.
inline hipError_t make_shape(bool two_d, uint64_t nx, uint64_t ny, uint64_t nz, uint32_t bx, uint32_t by,
                             uint32_t bz, LaunchShape& s) {
    if (bx == 0 || by == 0 || bz == 0) return hipErrorInvalidConfiguration;
    if (two_d) {
        nz = 1;
        bz = 1;
    }
    if (nx == 0 || ny == 0 || nz == 0) return hipErrorInvalidValue;
    if (static_cast<uint64_t>(bx) * by * bz > 1024) return hipErrorInvalidConfiguration;
    // Cell numbers are 32-bit, with room for a grid-stride step of the
    // statistics kernels (kMaxCells + 2^18 < 2^32); each factor and partial
    // product is checked first, so nothing overflows.
    if (nx > kMaxExtent || ny > kMaxExtent || nz > kMaxExtent) return hipErrorInvalidValue;
    if (nx * ny > kMaxCells || nx * ny * nz > kMaxCells) return hipErrorInvalidValue;
    const uint32_t threads = bx * by * bz;
    const uint64_t count = nx * ny * nz;
    if ((count + threads - 1) / threads > kMaxBlocks) return hipErrorInvalidConfiguration;
    s.block = dim3(threads, 1, 1);
    s.grid = dim3(static_cast<unsigned>((count + threads - 1) / threads), 1, 1);
    s.nx = static_cast<int>(nx);
    s.ny = static_cast<int>(ny);
    s.nz = static_cast<int>(nz);
    s.cells = Cells{static_cast<uint32_t>(nx), static_cast<uint32_t>(ny), static_cast<uint32_t>(nz),
                    static_cast<uint32_t>(count), make_fastdiv(static_cast<uint32_t>(nx)),
                    make_fastdiv(static_cast<uint32_t>(ny)), 0u, static_cast<uint32_t>(ny), 1u,
                    make_fastdiv(static_cast<uint32_t>(ny)), kDispatchOrder};
    return hipSuccess;
}

// Dense tiles of `rows` rows for population buffers: 0 = the reference's
// planes (plane = cells, zgap = 0); otherwise each tile holds the Q planes of
// its cells back to back, so the plane stride is the tile's cell count and
// zgap = (Q - 1) x that.  rows divides ny (rows = ny in 3D: the slab order
// [Z][Q][Y][X]).  Sets the shape's tiles and the largest Q's gap (a buffer of
// q planes has gap (q - 1) plane) and returns the plane stride.  The lanes'
// offsets must stay below 2^32 elements for the largest Q.
inline hipError_t tile_layout(bool two_d, uint64_t rows, int q_max, LaunchShape& s, uint64_t& plane) {
    (void)two_d;
    Cells& c = s.cells;
    if (rows == 0) {
        plane = c.count;
        return hipSuccess;
    }
    if (c.ny % rows != 0) return hipErrorInvalidValue;
    plane = static_cast<uint64_t>(c.nx) * rows;
    c.rows = static_cast<uint32_t>(rows);
    c.tiles = static_cast<uint32_t>(c.ny / rows);
    c.by_rows = make_fastdiv(static_cast<uint32_t>(rows));
    if (static_cast<uint64_t>(q_max) * c.count > 0xFFFFFFFFull) return hipErrorInvalidValue;
    c.zgap = static_cast<uint32_t>((q_max - 1) * plane);
    return hipSuccess;
}

inline uint64_t address(const void* p) { return reinterpret_cast<uint64_t>(p); }

inline hipStream_t as_stream(void* s) { return static_cast<hipStream_t>(s); }

// Residency cap for the memory-bound 3D fluid kernels.  They need few
// registers (45-50 VGPRs), so the hardware keeps 8 waves per SIMD (32 per CU)
// resident; with 19-27 population streams per wave that many outstanding
// streams run the HBM below its best rate.  Reserving LDS the kernels do not
// use caps the blocks per CU: at 16 waves per CU the D3Q19 TRT FP32 step at
// 256^3 ran 4.7% faster (39.1k against 37.3k MLUPS), 512^3 ~10%, D3Q27 TRT
// FP32 and FP16 (deviation form) ~4%; 20 waves per CU gave the same, 24
// less, 12 lost ground.  Kernels whose collision keeps the VALU busy
// (reference-order FP16/BF16) lose from it, as did the 2D fused reactive
// step, so the launchers apply it per kernel.
constexpr uint32_t kCappedWavesPerCu = 16;

// LDS per CU and per block of the current device (queried once per device).
struct LdsLimits {
    uint32_t per_cu = 0, per_block = 0;
};

inline LdsLimits lds_limits() {
    static LdsLimits cache[64];
    static std::once_flag once[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return LdsLimits{};
    std::call_once(once[dev], [dev] {
        int cu = 0, block = 0;
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) == hipSuccess &&
            hipDeviceGetAttribute(&block, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
            cu > 0 && block > 0)
            cache[dev] = LdsLimits{static_cast<uint32_t>(cu), static_cast<uint32_t>(block)};
    });
    return cache[dev];
}

// Dynamic LDS bytes per block that hold a launch of `threads`-wide blocks to
// `waves` resident waves per CU (0: no cap, e.g. blocks of more than half
// that many waves, or a device whose limits could not be read).
inline uint32_t capped_lds(uint32_t threads, uint32_t waves = kCappedWavesPerCu) {
    const uint32_t blocks = waves / ((threads + 63) / 64);
    if (blocks < 2) return 0;
    const LdsLimits l = lds_limits();
    const uint32_t lds = l.per_cu / blocks;
    return (lds == 0 || lds > l.per_block) ? 0 : lds;
}

// The dispatcher hands workgroup b to XCD b % 8 (8 XCDs, each with its own
// L2).  Blocks numbered linearly over the cells share the cache lines at their
// x edges with their neighbours, so in that dispatch order every edge line is
// fetched into two L2s (+6.6% of the reads of a 2D FP32 reactive step at
// 2048^2, +13% in FP16: rocprofv3 FETCH_SIZE), and an edge line that two
// blocks write leaves two L2s in parts.  Renumbering the blocks gives each XCD
// runs of consecutive ones.  kContiguousOrder: one run per XCD (a bijection
// for any grid size: XCDs x < nb % 8 take one block more).  1 <= order < 31:
// runs of 2^order blocks, eight runs (one per XCD) after another; the blocks
// past the last whole group of eight runs keep the dispatch order.
// The block that the dispatcher's block b of nb works on.
__host__ __device__ __forceinline__ uint32_t block_at(uint32_t b, uint32_t nb, uint32_t order) {
    if (order == kDispatchOrder) return b;
    if (order == kContiguousOrder) {
        const uint32_t q = nb / kXcds, r = nb % kXcds;
        const uint32_t x = b % kXcds, slot = b / kXcds;
        return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + slot;
    }
    const uint32_t group = kXcds << order;
    const uint32_t first = b & ~(group - 1u);
    if (nb - first < group) return b;
    const uint32_t r = b - first;
    return first + ((r % kXcds) << order) + r / kXcds;
}

__device__ __forceinline__ uint32_t ordered_block(uint32_t order) { return block_at(blockIdx.x, gridDim.x, order); }

// How a launch moves its populations: streaming or ordinary stores, and the
// order of its blocks.
struct Traffic {
    bool streaming;
    uint32_t order;
};

// Two levels of populations up to the size of the memory-side cache (256 MiB)
// stay there from one step of a time loop to the next, so ordinary stores win.
// D3Q19 TRT, streaming -> ordinary: 64^3 FP64 (80 MB) 16.1 -> 13.1 us, 112^3
// FP32 (213 MB) 46.1 -> 33.9 us; 2D FP32 512^2 5.8 -> 3.9 us, 1448^2 (151 MB)
// 28.2 -> 22.8 us.  Above it they gain little or lose: 128^3 FP32 (319 MB) 62.5
// -> 58.3 us, 112^3 FP64 (427 MB) 79.8 -> 82.1 us, 160^3 FP32 (623 MB) 116 ->
// 120 us, 256^3 FP32 425 -> 450 us, and a step whose output is not read next
// pays for what they displace (128^3 FP32 47 -> 61 us).
constexpr uint64_t kCachedBytes = 256ull << 20;

// Streaming stores need every wave to write whole 64-byte sectors: the planes
// `plane` elements apart and the base both on multiples of 64 bytes.  Where
// they are not, each wave writes parts of two lines per plane, and a streaming
// store sends them on before the neighbouring wave's part arrives: D3Q27 TRT
// FP32 at 253 x 191 x 167 ran 427 us against 385 us with ordinary stores, and
// 346 us with the blocks also in runs of 32 (the parts at the blocks' edges
// then meet in one L2); D3Q19 TRT FP16 at 301 x 217 x 185 271, 230 and 194 us.
//
// The order, by what was measured (256-work-item blocks):
//  - ordinary stores, 3D: runs of 32 (runs of 8 to 64 are within 2%).
//  - 2D up to kContiguousBytes: contiguous, with either store (in the caches
//    D2Q9 FP64 at 512^2 9.2 us in dispatch order, 7.1 us; FP32 at 1001 x 701 10.3
//    -> 9.0 us; past them FP32 at 2048^2, 288 MiB, 62.6 us in dispatch order,
//    61.0 in runs of 8, 55.0 contiguous; FP64 at 1448^2 58.4 -> 54.0 us).
//  - ordinary stores, larger 2D: runs of 32 (FP32 at 4095 x 2047 120 -> 109 us,
//    contiguous 120).
//  - streaming stores, larger 2D: runs of 8 up to 4 bytes per element (FP32 at
//    4096 x 2048 107 us in dispatch order, 111 contiguous, 102 in runs) and FP64
//    in dispatch order (206 us, 210 in runs).
//  - streaming stores, 3D: FP32 in dispatch order (256^3 425 us, in runs of 8
//    446 us: each XCD's separate window of the 38 streams costs more than the
//    edge lines save), the other formats in runs of 8 (D3Q19 FP16 at 256^3 223
//    -> 212 us, BF16 at 256 x 256 x 200 193 -> 185 us, FP64 at 128^3 127 -> 118
//    us, at 192^3 level), but for planes in step (kPlanesInStep).
//
// bases: the addresses of the buffers written, ORed; footprint: the bytes of
// the buffers that the step's time loop reads and writes.
//
// kContiguousBytes: the memory-side cache and the eight L2s of 4 MiB hold 288
// MiB, and the measured line lies just above: contiguous still wins at 295 MiB
// (FP64 at 2093 x 1026 56 us, in runs of 32 59-62), loses a little at 297 (FP32
// at 2048 x 2112 56.6 us, in runs of 8 55.2) and much at 340 (FP32 at 2048 x 2304
// 71.9 and 60.7; FP64 at 1536^2 70.1, in dispatch order 61.6; FP16 at 3072^2 72.0
// and 60.2; ordinary stores, FP32 at 2201 x 2199 84.8, in runs of 32 67.4).
constexpr uint64_t kContiguousBytes = 296ull << 20;

// Planes a multiple of 256 MiB apart: the streams of one cell share their
// channels and cache sets, and in runs eight windows of them meet (D3Q19, each
// time in four placements of the buffers, runs of 8 against dispatch order: TRT
// FP16 at 512^3 1.86-2.27 against 1.81-1.92 ms, at 256 x 1024 x 512 1.93-2.06
// against 1.76-1.87, at 512 x 512 x 1024 4.45 against 3.85; MRT BF16 at 512^3
// 2.04-2.16 against 1.80-1.94; D3Q27 TRT FP16 2.69-3.10 against 2.61-2.82; FP64
// at 512 x 512 x 128 2.01-2.09 against 1.93-1.98).  Planes of 128 MiB go both
// ways by their shape (256 x 256 x 1024 FP16 0.90 against 0.92-0.98 ms, 1024 x
// 256 x 256 0.90-0.98 against 0.92-0.97), as do FP64 planes of 512 MiB (512 x
// 512 x 256 3.46-4.03 against 3.57-4.01).
constexpr uint64_t kPlanesInStep = 256ull << 20;

// 16-bit planes within 128 KiB of a small multiple of 4 MiB lose in runs too
// (D3Q19 TRT FP16 / BF16, runs of 8 over dispatch order in three placements: 8 MiB
// 1.06-1.14 / 1.04-1.18, 11.9 1.09-1.13 / 1.00-1.07, 12 1.03-1.07, 16 1.04 / 1.05, 20
// 1.01-1.04 / 1.00-1.06, 24 0.99-1.07 / 0.98-1.04; D3Q27 FP16 8 MiB 1.03-1.08, 12
// 1.00-1.03; between them, 7.75 to 23 MiB, 0.97-0.99, and 28 MiB and more 0.96-0.99).
constexpr uint64_t kStepNear = 128ull << 10, kStepMost = 25ull << 20;

inline bool planes_in_step(uint64_t bytes, uint64_t element) {
    constexpr uint64_t kStep = 4ull << 20;
    if (element == 2 && bytes + kStepNear >= kStep && bytes < kStepMost && (bytes + kStepNear) % kStep <= 2 * kStepNear)
        return true;
    return bytes % kPlanesInStep == 0 && (element == 2 || bytes == kPlanesInStep);
}

// The order past the caches, of planes `plane` elements apart.
template <int D, class S> uint32_t large_order(bool streaming, uint64_t plane) {
    if (!streaming) return 5u;
    if (D == 2) return sizeof(S) <= 4 ? 3u : kDispatchOrder;
    return sizeof(S) == 4 || planes_in_step(plane * sizeof(S), sizeof(S)) ? kDispatchOrder : 3u;
}

template <int D, class S>
Traffic plan_traffic(const LaunchShape& s, uint64_t bases, uint64_t plane, uint64_t footprint) {
    const uint64_t misaligned = (bases | plane * sizeof(S) | static_cast<uint64_t>(s.cells.zgap) * sizeof(S)) % 64;
    const bool streaming = footprint > kCachedBytes && misaligned == 0;
    if (D == 2 && footprint <= kContiguousBytes) return Traffic{streaming, kContiguousOrder};
    return Traffic{streaming, large_order<D, S>(streaming, plane)};
}

}  // namespace lbc
