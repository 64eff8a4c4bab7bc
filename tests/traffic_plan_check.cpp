// Host check of the steps' store form and block order (the rules of
// lb-cube_amd/csrc/lbc_launch.hpp and lbc_reactive.hpp, the headers' own code).
// Each line of stdin is "<step> <element bytes> <nx> <ny> <nz> <Q> <offset>":
// step is fluid, slabs (the fluid step in the slab order), fused, reaction or
// scalar, Q the fluid's; the planes of a domain lie back to back, `offset` bytes
// past a cache line (nz = 1: 2D).
// Prints "<streaming> <order>" for each.
#include <cstdint>
#include <cstdio>
#include <cstring>

#include "../lb-cube_amd/csrc/lbc_launch.hpp"
#include "../lb-cube_amd/csrc/lbc_reactive.hpp"

template <int D, class T> lbc::Traffic plan(const char* step, lbc::LaunchShape& s, int q, uint64_t base) {
    const uint64_t qs = D == 2 ? 5 : 7;
    if (std::strcmp(step, "fused") == 0) return lbc::adr_traffic<D, T, lbc::kFusedStep>(s, false, base, 2 * q, 4 * qs);
    if (std::strcmp(step, "reaction") == 0) return lbc::adr_traffic<D, T, lbc::kReactionStep>(s, false, base, 2 * q, 4 * qs);
    if (std::strcmp(step, "scalar") == 0) return lbc::adr_traffic<D, T, lbc::kScalarStep>(s, false, base, 2 * q, 2 * qs);
    if (std::strcmp(step, "slabs") == 0) {
        const uint64_t cells = s.cells.count, slab = cells / s.cells.nz;
        s.cells.zgap = static_cast<uint32_t>((q - 1) * slab);
        return lbc::plan_traffic<D, T>(s, base, slab, 2ull * q * cells * sizeof(T));
    }
    return lbc::plan_traffic<D, T>(s, base, s.cells.count, 2ull * q * s.cells.count * sizeof(T));
}

template <int D> lbc::Traffic by_size(const char* step, int size, lbc::LaunchShape& s, int q, uint64_t base) {
    return size == 8   ? plan<D, double>(step, s, q, base)
           : size == 4 ? plan<D, float>(step, s, q, base)
                       : plan<D, uint16_t>(step, s, q, base);
}

int main() {
    char step[16];
    int size, q;
    unsigned long long nx, ny, nz, base;
    while (std::scanf("%15s %d %llu %llu %llu %d %llu", step, &size, &nx, &ny, &nz, &q, &base) == 7) {
        lbc::LaunchShape s;
        if (lbc::make_shape(nz == 1, nx, ny, nz, 256, 1, 1, s) != hipSuccess) return std::printf("FAIL shape\n"), 1;
        const lbc::Traffic t = nz == 1 ? by_size<2>(step, size, s, q, base) : by_size<3>(step, size, s, q, base);
        std::printf("%d %u\n", t.streaming ? 1 : 0, t.order);
    }
    return 0;
}
