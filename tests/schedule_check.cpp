// Host check of the gradient's schedule (lbc_trajectory.hpp, the header's own
// code).  Each line of stdin is "<dim> <Q fluid> <Q species> <compact> <steps>
// <interval> <cells> <element bytes> <paired>"; prints "<segment length>
// <segments> <first segment's steps> <overlapped>" for each.
#include <cstdio>

#include "../lb-cube_amd/csrc/lbc_trajectory.hpp"

int main() {
    unsigned long long dim, qf, qs, compact, steps, interval, cells, element, paired;
    while (std::scanf("%llu %llu %llu %llu %llu %llu %llu %llu %llu", &dim, &qf, &qs, &compact, &steps, &interval,
                      &cells, &element, &paired) == 9) {
        const std::size_t state = qf + 2 * qs;
        const lbc::TrajectoryPlan plan =
            lbc::plan_trajectory(lbc::trajectory_layout(compact != 0, dim, qf, qs), steps,
                                 lbc::trajectory_capacity(state, steps, interval));
        if (plan.length == 0) return std::printf("FAIL no plan\n"), 1;
        std::printf("%zu %zu %zu %d\n", plan.length, plan.segments, plan.first(steps),
                    lbc::overlapped(plan, state * cells * element, dim, element, paired != 0) ? 1 : 0);
    }
    return 0;
}
