// One cell of the fused fluid + A + B -> C reactive step (shared by the
// single-domain and the ensemble kernels).
#pragma once

#include "lbc_fast.hpp"
#include "lbc_launch.hpp"
#include "lbc_physics.hpp"
#include "lbc_storage.hpp"

namespace lbc {

// Where one cell's populations come from: `pf` locates the cell and its
// periodic sources in the fluid planes and `ps` in the species planes (the
// same pull unless the buffers are stored in tiles, whose gaps differ with the
// lattices' Q), `plane` is the element stride between population planes; WIDE
// selects 64-bit per-lane addresses (planes of more than 4 GiB).
template <class F, class S, class T, bool WIDE> struct CellSources {
    const T *__restrict__ cf, *__restrict__ ca, *__restrict__ cb;
    const Pull &pf, &ps;
    size_t plane;
    __device__ __forceinline__ const T* f(int i) const {
        return at<WIDE>(plane_ptr(cf, i, plane), pf.src(F::cx[i], F::cy[i], F::cz[i]));
    }
    __device__ __forceinline__ const T* a(int i) const {
        return at<WIDE>(plane_ptr(ca, i, plane), ps.src(S::cx[i], S::cy[i], S::cz[i]));
    }
    __device__ __forceinline__ const T* b(int i) const {
        return at<WIDE>(plane_ptr(cb, i, plane), ps.src(S::cx[i], S::cy[i], S::cz[i]));
    }
};

// Where they go: the cell's element offsets in the fluid and species planes.
template <class T, bool WIDE> struct CellTargets {
    T *__restrict__ nf, *__restrict__ na, *__restrict__ nb;
    uint32_t cell, scell;
    size_t plane;
    __device__ __forceinline__ T* f(int i) const { return at<WIDE>(plane_ptr(nf, i, plane), cell); }
    __device__ __forceinline__ T* a(int i) const { return at<WIDE>(plane_ptr(na, i, plane), scell); }
    __device__ __forceinline__ T* b(int i) const { return at<WIDE>(plane_ptr(nb, i, plane), scell); }
};

// Fluid step + A + B -> C step of one cell: populations read through `in` and
// stored through `out` (CellSources and CellTargets, or a tile in LDS); NT: the
// store form.
// The reaction step of the reference reads the fluid populations that the
// fluid step has just written
// at the same cell (src/simulate_reaction.cpp:527-541); here they are still in
// registers.  With reduced-precision storage they are passed through the
// storage rounding first, so the velocity is the one the unfused pair sees.
// Shared by the single-domain, ensemble and gradient kernels.  Returns the
// density and velocity of the new fluid state.
template <class F, int CT, class S, int ST, bool NT, class In, class Out>
__device__ __forceinline__ Macro<typename Storage<ST>::R> reactive_update(
    const In& in, const Out& out, typename Storage<ST>::R omega, typename Storage<ST>::R omega_minus,
    typename Storage<ST>::R omega_c, typename Storage<ST>::R k_react, typename Storage<ST>::R ref_a,
    typename Storage<ST>::R ref_b) {
    using St = Storage<ST>;
    using R = typename St::R;
    R f[F::Q];
#pragma unroll
    for (int i = 0; i < F::Q; ++i) f[i] = St::load(in.f(i), kOffsetStorage<ST> ? R(F::w[i]) : R(0));
    collide_cell<F, CT, R>(f, omega, omega_minus, [&](int i, R v) {
        St::template store<NT>(out.f(i), v, kOffsetStorage<ST> ? R(F::w[i]) : R(0));
    });
    if constexpr (kOffsetStorage<ST>) {
#pragma unroll
        for (int i = 0; i < F::Q; ++i) f[i] = St::roundtrip(f[i], R(F::w[i]));
    }
    const Macro<R> m = macro_state<F, R>(f);
    R ga[S::Q], gb[S::Q];
#pragma unroll
    for (int i = 0; i < S::Q; ++i) {
        ga[i] = St::load(in.a(i), R(S::w[i]) * ref_a);
        gb[i] = St::load(in.b(i), R(S::w[i]) * ref_b);
    }
    const R ca = concentration<S, R>(ga);
    const R cb = concentration<S, R>(gb);
    const R source = reaction_source<R>(ca, cb, k_react);
    collide_scalar<S, R>(ga, m.ux, m.uy, m.uz, omega_c, source);
    collide_scalar<S, R>(gb, m.ux, m.uy, m.uz, omega_c, source);
#pragma unroll
    for (int i = 0; i < S::Q; ++i) {
        St::template store<NT>(out.a(i), ga[i], R(S::w[i]) * ref_a);
        St::template store<NT>(out.b(i), gb[i], R(S::w[i]) * ref_b);
    }
    return m;
}

// The same step in the deviation form (LBC_FLAG_FAST; BGK, TRT, MRT): fluid
// populations carried as f_i - w_i with FMAs and a hardware reciprocal
// (lbc_fast.hpp), the velocity taken from the deviations as stored, the scalar
// collision with 1/cs2 multiplied and the rest equilibrium by remainder, the
// reaction increment without cancellation (lbc_fast.hpp).
template <class F, int CT, class S, int ST, bool NT, class In, class Out>
__device__ __forceinline__ Macro<typename Storage<ST>::R> reactive_update_fast(
    const In& in, const Out& out, typename Storage<ST>::R omega, typename Storage<ST>::R omega_minus,
    typename Storage<ST>::R omega_c, typename Storage<ST>::R k_react, typename Storage<ST>::R ref_a,
    typename Storage<ST>::R ref_b) {
    using St = Storage<ST>;
    using R = typename St::R;
    R d[F::Q];
#pragma unroll
    for (int i = 0; i < F::Q; ++i) d[i] = St::load_dev(in.f(i), R(F::w[i]));
    collide_dev<F, CT, R>(d, omega, omega_minus,
                          [&](int i, R v) { St::template store_dev<NT>(out.f(i), v, R(F::w[i])); });
#pragma unroll
    for (int i = 0; i < F::Q; ++i) d[i] = St::roundtrip_dev(d[i], R(F::w[i]));
    const DevMacro<F, R> m = dev_macro<F, R>(d);
    R ga[S::Q], gb[S::Q];
#pragma unroll
    for (int i = 0; i < S::Q; ++i) {
        ga[i] = St::load(in.a(i), R(S::w[i]) * ref_a);
        gb[i] = St::load(in.b(i), R(S::w[i]) * ref_b);
    }
    const R ca = concentration<S, R>(ga);
    const R cb = concentration<S, R>(gb);
    const R source = reaction_source_fast<R>(ca, cb, k_react);
    collide_scalar_fast<S, R>(ga, ca, m.ux, m.uy, m.uz, omega_c, source);
    collide_scalar_fast<S, R>(gb, cb, m.ux, m.uy, m.uz, omega_c, source);
#pragma unroll
    for (int i = 0; i < S::Q; ++i) {
        St::template store<NT>(out.a(i), ga[i], R(S::w[i]) * ref_a);
        St::template store<NT>(out.b(i), gb[i], R(S::w[i]) * ref_b);
    }
    return Macro<R>{m.rho, m.ux, m.uy, m.uz};
}

template <class F, int CT, class S, int ST, bool WIDE = false, bool NT = true>
__device__ __forceinline__ Macro<typename Storage<ST>::R> reactive_cell(
    const typename Storage<ST>::S* __restrict__ cur_f, typename Storage<ST>::S* __restrict__ nxt_f,
    const typename Storage<ST>::S* __restrict__ cur_a, typename Storage<ST>::S* __restrict__ nxt_a,
    const typename Storage<ST>::S* __restrict__ cur_b, typename Storage<ST>::S* __restrict__ nxt_b, const Pull& pf,
    const Pull& ps, size_t plane, typename Storage<ST>::R omega, typename Storage<ST>::R omega_minus,
    typename Storage<ST>::R omega_c, typename Storage<ST>::R k_react, typename Storage<ST>::R ref_a,
    typename Storage<ST>::R ref_b) {
    using T = typename Storage<ST>::S;
    return reactive_update<F, CT, S, ST, NT>(CellSources<F, S, T, WIDE>{cur_f, cur_a, cur_b, pf, ps, plane},
                                CellTargets<T, WIDE>{nxt_f, nxt_a, nxt_b, pf.dst, ps.dst, plane}, omega,
                                omega_minus, omega_c, k_react, ref_a, ref_b);
}

template <class F, int CT, class S, int ST, bool WIDE = false, bool NT = true>
__device__ __forceinline__ Macro<typename Storage<ST>::R> reactive_cell_fast(
    const typename Storage<ST>::S* __restrict__ cur_f, typename Storage<ST>::S* __restrict__ nxt_f,
    const typename Storage<ST>::S* __restrict__ cur_a, typename Storage<ST>::S* __restrict__ nxt_a,
    const typename Storage<ST>::S* __restrict__ cur_b, typename Storage<ST>::S* __restrict__ nxt_b, const Pull& pf,
    const Pull& ps, size_t plane, typename Storage<ST>::R omega, typename Storage<ST>::R omega_minus,
    typename Storage<ST>::R omega_c, typename Storage<ST>::R k_react, typename Storage<ST>::R ref_a,
    typename Storage<ST>::R ref_b) {
    using T = typename Storage<ST>::S;
    return reactive_update_fast<F, CT, S, ST, NT>(CellSources<F, S, T, WIDE>{cur_f, cur_a, cur_b, pf, ps, plane},
                                     CellTargets<T, WIDE>{nxt_f, nxt_a, nxt_b, pf.dst, ps.dst, plane}, omega,
                                     omega_minus, omega_c, k_react, ref_a, ref_b);
}

// Residency cap (kCappedWavesPerCu, lbc_launch.hpp), measured on the 256^3
// TGV with two D3Q7 species.  FP32: scalar step 41.2k -> 45.0k MLUPS,
// reaction step 30.9k -> 31.8k, fused TRT step 21.0k -> 21.3k (both forms).
// FP16: the fused step gains 3-4.5% (39.2k -> 40.4k, deviation form 39.3k ->
// 41.1k), the scalar step loses 7%, the reaction step gains 1.4% (left
// uncapped).  BF16 loses up to 15% and FP64 is unchanged, so both stay
// uncapped, as do 2D grids (the fused 2048^2 step lost 1-5%).
template <int D, int ST, bool FUSED> constexpr bool capped_residency_adr() {
    return D == 3 && (ST == kF32 || (FUSED && ST == kF16));
}

// The memory-side cache has 16 ways of 16 MiB.  Where a small multiple of the
// plane (q of them) is a multiple of 16 MiB, every q-th plane falls on the same
// sets; from planes / q > 16 streams on they crowd the ways, and a grid whose
// blocks all work on one window of each plane loses what the cache held.  A
// contiguous run per XCD spreads each plane over eight windows.  The least such
// q up to 4, or 0.
inline uint64_t crowding(uint64_t plane_bytes, uint64_t planes) {
    constexpr uint64_t kWay = 16ull << 20, kNear = kWay / 64;
    for (uint64_t q = 1; q <= 4 && planes > 16 * q; ++q) {
        const uint64_t end = q * plane_bytes + kNear;
        if (end >= kWay && end % kWay <= 2 * kNear) return q;
    }
    return 0;
}

// The store form and the block order of a step whose time loop holds `fluid`
// and `species` population planes and that writes at `bases`.  Loops in the
// caches follow plan_traffic, tiled buffers and planes of more than 4 GiB stream
// in dispatch order.  Past the caches the general order holds (large_order), but
// crowded planes run contiguously up to kCrowdedBytes (us, three placements of
// the buffers or more, general order -> contiguous):
//  - fused, crowded: D2Q9 MRT FP32 2048^2 109-140 -> 107-118; FP64 2048 x 1024
//    122-130 -> 109-114; FP16 4096 x 2048 118-124 -> 113-122; D3Q19 TRT FP32 128^3
//    99-111 -> 94-104, 112^3 69-79 -> 64-70.
//  - fused, not crowded: 1920^2 FP32 104 -> 125, 3072^2 FP16 135 -> 153, FP64
//    1152^2 74 -> 82; D3Q19 FP32 120^3 85 -> 94, 136^3 119.5 -> 130, FP16 168^3 123
//    -> 149; D3Q27 FP32 120^3 106 -> 117.
//  - crowded past the limit: 2048 x 4096 FP32 229 -> 241; D3Q19 FP16 192 x 256 x
//    128 161 -> 170, FP32 256 x 128 x 128 195-198 -> 194-204.
//  - 3D at 2 bytes, where q < 3 gains nothing: in dispatch order (TRT FP16 256 x
//    256 x 64 100 us, contiguous 101; BF16 512 x 128 x 64 108 and 109).
constexpr uint64_t kCrowdedBytes = 730ull << 20;

// The launch of the species alone reads what the fluid's launch has left.  2D:
// in the fluid's order while that is contiguous (D2Q9 and two species, FP64 at
// 1472^2, loop of two launches: both contiguous 143.6 us, both in dispatch
// order 139.7, one of each 148.8).  3D: contiguous where crowded up to
// kCrowdedSpecies (D3Q19 FP32 256 x 128 x 128 247-257 -> 239-247, FP64 128^3
// 253-275 -> 242-253).  Else FP64 in runs of 8 up to kSpeciesRuns64 (120^3 214.8
// -> 210.5) and in dispatch order above (256^3 2028-2046, in runs 2081-2098; 256 x
// 256 x 192 1578 and 1681), FP32 so with kSpeciesRuns32 (104^3 61.1 -> 59.6, two
// scalars at 120^3 112 -> 107; 128 x 128 x 112 110.5 and 111.7), 2-byte storage in
// dispatch order (FP16 320^3 1004-1018, in runs 1058-1075, with two scalars 1215
// and 1271; from 144^3 to 416^3 else within 2% either way).
// Misaligned 2D planes: streaming stores leave the fluid in the caches.
// Contiguous up to kSpeciesStream (ordinary -> streaming: two scalars FP32 1801
// x 1799 120 -> 115, FP64 1301 x 1299 129 -> 121; reaction FP64 1201 x 1199 107 ->
// 97) and, one species at a time, where crowded (two scalars FP32 2049 x 2047
// 185 -> 165, FP64 1449 x 1447 178 -> 157; the reaction step FP32 2049 x 2047 157
// with ordinary stores, 161 streaming), then FP64 scalars in dispatch order up
// to kSpeciesStream64 (1501 x 1499 181 -> 173, 1551 x 1549 194 -> 185; not the
// reaction step: 1301 x 1299 118 -> 123, nor FP32 and FP16: 2401 x 2399 240 -> 248,
// 3001 x 2999 189 -> 195).
constexpr uint64_t kCrowdedSpecies = 1100ull << 20, kSpeciesRuns64 = 730ull << 20, kSpeciesRuns32 = 450ull << 20;
constexpr uint64_t kSpeciesStream = 420ull << 20, kSpeciesStream64 = 560ull << 20;

enum AdrLaunch { kFusedStep, kReactionStep, kScalarStep };

template <int D, class T, AdrLaunch L>
Traffic adr_traffic(LaunchShape& s, bool tiled, uint64_t bases, uint64_t fluid, uint64_t species) {
    constexpr bool fused = L == kFusedStep;
    const uint64_t plane = s.cells.count, bytes = plane * sizeof(T), loop = (fluid + species) * bytes;
    Traffic t = plan_traffic<D, T>(s, bases, plane, loop);
    if (tiled || wide_planes<T>(s)) {
        t = Traffic{true, kDispatchOrder};
    } else if (loop > kCachedBytes) {
        const uint64_t q = crowding(bytes, fluid + species);
        const bool crowded = q != 0 && loop <= (fused || D == 2 ? kCrowdedBytes : kCrowdedSpecies);
        t.order = large_order<D, T>(t.streaming, plane);
        if (crowded && (D == 2 || (t.streaming && (sizeof(T) > 2 || q > 2)))) t.order = kContiguousOrder;
        if (!fused && D == 2) {
            if (t.streaming && fluid * bytes <= kContiguousBytes) t.order = kContiguousOrder;
            if (!t.streaming && ((crowded && L == kScalarStep) || loop <= kSpeciesStream))
                t = Traffic{true, kContiguousOrder};
            if (!t.streaming && L == kScalarStep && sizeof(T) == 8 && loop <= kSpeciesStream64)
                t = Traffic{true, kDispatchOrder};
        }
        if (!fused && D == 3 && t.streaming && !crowded) {
            constexpr uint64_t runs = sizeof(T) == 8 ? kSpeciesRuns64 : sizeof(T) == 4 ? kSpeciesRuns32 : 0;
            t.order = loop <= runs ? 3u : kDispatchOrder;
        }
    }
    s.cells.order = t.order;
    return t;
}

}  // namespace lbc
