// group_steps.hpp -- step words of the group sweeps' barrier (plain C++, so that
// the host can test the comparisons).
//
// Steps count on from launch to launch, and a launch refreshes only the words
// of the workgroups that take part in it: a word may be any number of steps
// behind when a launch begins.  Words of 64 bits never wrap (2^64 steps of
// 0.3 us), so one that lies behind compares as behind for good; in 32 bits one
// 2^31 steps behind (half an hour of sweeps) would pass as ahead, and its
// barrier with it.  A launch therefore meets on words of 64 bits before its
// first step.  The words of its steps have 32 bits (32 of them share a cache
// line; 64 bits there cost the sweeps on all XCDs 1.4% of a solve): each was
// set to the step before the launch's first by its owner, before that came to
// the meeting, so it lies within the launch's own steps, which are fewer than
// 2^31.
#pragma once

namespace unap_hip {

using GroupStep = unsigned long long;
constexpr bool groupReached(GroupStep word, GroupStep step) { return word >= step; }
constexpr bool groupReached(unsigned word, unsigned step) { return (int)(word - step) >= 0; }

// The top bit of the steps' count says that a wait has given up.
constexpr GroupStep kGroupBroken = 1ull << 63;
constexpr bool groupBroken(GroupStep epoch) { return (epoch & kGroupBroken) != 0; }

// Gauss-Seidel sweeps of nl levels, of `left` still to do, that one launch
// takes: at most 2^20 steps (far below 2^31; about a second), or one sweep.
constexpr int kGroupSteps = 1 << 20;
constexpr int groupSweeps(int nl, int left) {
    const int most = nl < kGroupSteps ? kGroupSteps / nl : 1;
    return left < most ? left : most;
}

}  // namespace unap_hip
