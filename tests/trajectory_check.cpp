// Host check of the gradient's trajectory plan (lbc_trajectory.hpp, the
// header's own code): for every run of up to 200 steps and interval of up to
// 210, compact or not, the plan fits the workspace, covers the steps and runs
// no more of them twice than segments of `interval` steps would.  Prints "ok
// <plans>" or the first failure.
#include <cstdio>

#include "../lb-cube_amd/csrc/lbc_trajectory.hpp"

int main() {
    const std::size_t lattices[3][3] = {{2, 9, 5}, {3, 19, 7}, {3, 27, 7}};
    std::size_t plans = 0;
    for (const auto& l : lattices)
        for (int compact = 0; compact < 2; ++compact) {
            const lbc::TrajectoryPlanes p = lbc::trajectory_layout(compact, l[0], l[1], l[2]);
            for (std::size_t steps = 1; steps <= 200; ++steps)
                for (std::size_t interval = 1; interval <= 210; ++interval, ++plans) {
                    const std::size_t capacity = lbc::trajectory_capacity(l[1] + 2 * l[2], steps, interval);
                    const lbc::TrajectoryPlan plan = lbc::plan_trajectory(p, steps, capacity);
                    const bool covers = plan.length > 0 && plan.first(steps) >= 1 && plan.first(steps) <= plan.length;
                    const bool fits = covers && lbc::trajectory_planes(p, steps, plan.length) <= capacity;
                    const std::size_t twice = steps > 2 * plan.length ? steps - 2 * plan.length : 0;
                    if (!fits || twice > (steps > 2 * interval ? steps - 2 * interval : 0))
                        return std::printf("FAIL q=%zu compact=%d steps=%zu interval=%zu length=%zu\n", l[1], compact,
                                           steps, interval, plan.length), 1;
                }
        }
    std::printf("ok %zu\n", plans);
    return 0;
}
