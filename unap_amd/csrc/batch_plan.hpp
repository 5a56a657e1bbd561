// batch_plan.hpp -- which systems of a batch teams of workgroups take, and how
// many teams (plain C++, so that the host can test it).
//
// A team of s workgroups on one XCD solves a system faster than one workgroup
// does, but not s times (teamSpeed), and while the whole chip is busy the
// difference is lost.  So teams pay only for the systems that one workgroup
// would still be solving when the rest of the chip has run out of work: those
// whose cost is above kTeamShare times a workgroup's share of all.  The teams
// hold as many workgroups as their share of the workgroups' time; the others
// take the other systems alone, and a team whose systems are taken joins them.
// ms a solve, one workgroup a system / this rule (MI355X, boxes with random
// numberings of the given edges; in brackets teams of 4 and of 8 for every
// system they can share): 96 of 8..48 367 / 131 [175 / 129], 300 of 8..40
// 203 / 117 [142 / 230], 512 of 8..48 505 / 302 [406 / 597], 1500 of 8..48
// 717 / 711, 600 of 28..32 333 / 333 [528 / 778], one of 48 and 1000 of 8..12
// 305 / 83 [122 / 84], 64 of 8..24 25 / 25.
#pragma once

#include <algorithm>
#include <cmath>
#include <vector>

namespace unap_hip {

constexpr int kTeamMax = 8;
// Workgroups worth having on a system of `rows` rows a level: a level's barrier
// costs a team about as much as one workgroup takes for kTeamRows rows of it.
constexpr int kTeamRows = 256;
constexpr int teamWant(int rows, int most) {
    const int want = (rows + kTeamRows - 1) / kTeamRows;
    return want < most ? want : most;
}

// How much faster a team of `size` solves a system than one workgroup does
// (random numberings, 768 / 1200 / 1820 / 3560 / 6140 rows a level: four
// workgroups 1.2 / 1.5 / 1.8 / 2.0 / 2.2, eight 1.1 / 1.6 / 2.1 / 2.8 / 3.0).
inline double teamSpeed(int size, int rows) {
    return 1.0 / (size > 4 ? 0.25 + 430.0 / rows : 0.42 + 260.0 / rows);
}
// Rows a level from which on teams are considered (below: 1.2 times at most,
// on an idle chip), and the share named above (1.0: 512 systems 316 ms, 150 of
// 24..40 188 against 168).
constexpr int kTeamLevelRows = 1024;
constexpr double kTeamShare = 1.25;

struct TeamSystem {
    int rows;     // a level, on average
    double cost;  // time in one workgroup, in arbitrary units
};
struct TeamPlan {
    int size = 1;  // workgroups a team; 1: none
    int wide = 0;  // systems for teams
    int teams = 0;
    std::vector<int> order;  // those, then the others, each in the order given
};

// order: the systems, largest first; forced: the size of the teams, which then
// take every system they can share (0: chosen).
inline TeamPlan planTeams(const std::vector<TeamSystem>& sys, const std::vector<int>& order, int cus, int forced) {
    TeamPlan p;
    p.order = order;
    if (forced == 1) return p;
    double all = 0.0;
    for (const TeamSystem& s : sys) all += s.cost;
    const auto mid = std::stable_partition(p.order.begin(), p.order.end(), [&](int i) {
        if (forced) return teamWant(sys[i].rows, forced) > 1;
        return sys[i].rows >= kTeamLevelRows && sys[i].cost > kTeamShare * all / cus;
    });
    p.wide = (int)(mid - p.order.begin());
    if (!p.wide) return p;
    double best = 0.0;
    for (const int s : {4, 8}) {
        const int size = forced ? forced : s;
        double longest = 0.0, time = 0.0, rest = all;  // of the teams' systems, their workgroups, the other systems
        for (int k = 0; k < p.wide; ++k) {
            const TeamSystem& w = sys[p.order[k]];
            const double t = w.cost / teamSpeed(size, std::max(1, w.rows));
            longest = std::max(longest, t);
            time += t * size;
            rest -= w.cost;
        }
        rest = std::max(rest, 0.0);
        const double estimate = longest + 1.2 * (time + rest) / cus;
        if (p.size > 1 && estimate >= best) break;
        best = estimate;
        p.size = size;
        p.teams = std::max(1, std::min({p.wide, cus / size, (int)std::ceil(cus * time / (time + rest) / size)}));
        if (forced) break;
    }
    return p;
}

}  // namespace unap_hip
