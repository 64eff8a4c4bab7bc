// Where the gradient keeps the forward trajectory: which steps' states stay,
// which are recomputed, and how the workspace holds them (host arithmetic).
#pragma once

#include <algorithm>
#include <cstddef>

namespace lbc {

// Steps 0..steps-1 are cut into segments of `length` steps, the first one
// shorter.  The sweep walks them last to first.  A step's slot holds what the
// sweep reads of it; two segment buffers of `length` slots take the segments
// in turn.  The forward run leaves the last two segments in them and a
// checkpoint at the start of every segment but the first (whose start is the
// caller's initial state); the other segments are run again, each into the
// buffer whose segment has been walked.  So all but 2 x `length` steps are
// run twice.
struct TrajectoryPlan {
    std::size_t length, segments;
    std::size_t first(std::size_t steps) const { return steps - (segments - 1) * length; }  // of segment 0
};

// Population planes of one checkpoint, one slot and the buffers beside them.
struct TrajectoryPlanes {
    std::size_t checkpoint, slot, scratch;
};

inline std::size_t trajectory_planes(const TrajectoryPlanes& p, std::size_t steps, std::size_t length) {
    const std::size_t segments = (steps + length - 1) / length;
    return (segments - 1) * p.checkpoint + std::min<std::size_t>(segments, 2) * length * p.slot + p.scratch;
}

// The longest segments that `capacity` planes hold (so the fewest steps are
// run twice); {0, 0} if none fit.
inline TrajectoryPlan plan_trajectory(const TrajectoryPlanes& p, std::size_t steps, std::size_t capacity) {
    for (std::size_t length = std::min(steps, capacity / p.slot); length > 0; --length)
        if (trajectory_planes(p, steps, length) <= capacity) return {length, (steps + length - 1) / length};
    return {0, 0};
}

// The workspace of a gradient in states of `state` planes: a checkpoint for
// each `interval` steps and two segments of `interval` states.
inline std::size_t trajectory_capacity(std::size_t state, std::size_t steps, std::size_t interval) {
    return ((steps + interval - 1) / interval + 2 * interval) * state;
}

// The planes of a run.  compact: a slot holds the density and velocity of the
// step's fluid (1 + dim planes) and the species it starts from; two fluid
// levels beside the slots; a checkpoint also carries the density and velocity
// of the step before it.  Else a slot holds the whole state.
inline TrajectoryPlanes trajectory_layout(bool compact, std::size_t dim, std::size_t qf, std::size_t qs) {
    if (!compact) return {qf + 2 * qs, qf + 2 * qs, 0};
    return {qf + 2 * qs + 1 + dim, 2 * qs + 1 + dim, 2 * qf};
}

}  // namespace lbc
