// Host check of the kernels' block order (block_at of
// lb-cube_amd/csrc/lbc_launch.hpp, the header's own code): for every grid size
// and order read from stdin the renumbering is a bijection of [0, nb), and in
// runs each XCD (b % 8) takes runs of 2^order consecutive blocks.  Prints
// "ok <grids>" or the first failure.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../lb-cube_amd/csrc/lbc_launch.hpp"

int main() {
    unsigned nb, order, grids = 0;
    while (std::scanf("%u %u", &nb, &order) == 2) {
        std::vector<char> seen(nb, 0);
        for (unsigned b = 0; b < nb; ++b) {
            const uint32_t t = lbc::block_at(b, nb, order);
            if (t >= nb || seen[t]) return std::printf("FAIL nb=%u order=%u b=%u -> %u\n", nb, order, b, t), 1;
            seen[t] = 1;
            if (order > 0 && order < 31 && t % (1u << order) != 0 && b >= 8 && t != b &&
                lbc::block_at(b - 8, nb, order) + 1 != t)
                return std::printf("FAIL run nb=%u order=%u b=%u\n", nb, order, b), 1;
        }
        ++grids;
    }
    std::printf("ok %u\n", grids);
    return 0;
}
