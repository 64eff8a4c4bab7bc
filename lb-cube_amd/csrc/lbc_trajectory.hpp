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

// Whether a segment is recomputed on a second stream while the caller's walks
// the next one: from three segments on (the last two are never recomputed) of
// at least kOverlapSteps steps (two cross-stream waits each), for states up to
// kOverlapMax: larger ones fill the GPU or displace each other from the caches
// (FP32 D2Q9 512^2, 1024 steps, 21.95 ms overlapped, 22.45 not; 1024^2, 256
// steps, 21.6 and 19.0; FP64 600^2, 200 steps, 10.6 and 10.4).  Down to the
// smallest states it pays, where the sweep's launches leave the GPU idle (BGK
// FP32 400 steps, interval 16, paired: 8^2 3.13 and 3.25 ms, 96^2 3.57 and 3.97,
// 200^2 3.67 and 4.22; RLBM FP64 1024 steps, interval 32: 64^2 12.4 and 15.1;
// D3Q19 RLBM FP32 300 steps: 16^3 3.95 and 5.0), except that the host cannot
// feed two streams with steps shorter than a launch: single 2D steps of FP32
// states below kShortState32 (FP64: kShortState64) need segments of
// kShortSteps (RLBM FP32 400 steps, interval 16: 128^2 5.15 and 4.53, 200^2 4.92
// and 4.91, 240^2 4.75 and 5.17; interval 32, 1024 steps: 128^2 12.1 and 13.0;
// FP64, interval 16: TRT 32^2 5.33 and 5.01, 64^2 5.23 and 5.25, RLBM 32^2 5.42 and
// 5.33, 64^2 5.34 and 5.56).
constexpr std::size_t kOverlapSteps = 8, kShortSteps = 32, kOverlapMax = 40u << 20;
constexpr std::size_t kShortState32 = 4u << 20, kShortState64 = 256u << 10;

// state_bytes: of one state of `element`-byte populations; paired: two steps
// per launch.
inline bool overlapped(const TrajectoryPlan& plan, std::size_t state_bytes, std::size_t dim, std::size_t element,
                       bool paired) {
    const bool brief = dim == 2 && !paired && state_bytes < (element == 4 ? kShortState32 : kShortState64);
    return plan.segments > 2 && plan.length >= (brief ? kShortSteps : kOverlapSteps) && state_bytes <= kOverlapMax;
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
