// joint_schedule.hpp -- the order in which the joint stage's solves run.
//
// The reference sweeps the joints in arena order, joint_iterations times
// (physics.rs:424-477): a solve reads and writes its two bodies' positions, so
// only solves that share a body have to keep their order.  A group of joints
// gets levels: every solve of every iteration in the first level after the
// latest one that touches one of its bodies, at most one wave's lanes of them
// a level.  A wave that runs a group's levels in turn, a lane a solve, gives
// the sequential sweep's very positions in as many dependent steps as there
// are levels -- against one step for each solve of the largest component when
// a lane sweeps a component alone.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <utility>
#include <vector>

namespace bg {

struct JointSchedule {
    std::vector<uint32_t> group_level{0};  // levels of group g: [group_level[g], group_level[g + 1])
    std::vector<uint32_t> level_start{0};  // solves of level l: entry[level_start[l] .. level_start[l + 1])
    std::vector<uint32_t> entry;           // a solve's joint
    std::vector<uint32_t> iteration;       // and its iteration

    uint32_t groups() const { return (uint32_t)group_level.size() - 1; }

    // Appends a group: `joints` in arena order (body a, body b of each, by any numbering below
    // n_bodies), numbered `ids`, swept `iterations` times.  `last` is scratch, all zero.
    void add_group(const std::vector<std::pair<uint32_t, uint32_t>>& joints, const std::vector<uint32_t>& ids,
                   uint32_t iterations, std::vector<uint32_t>& last, uint32_t width) {
        std::vector<std::vector<std::pair<uint32_t, uint32_t>>> levels;
        for (uint32_t it = 0; it < iterations; ++it)
            for (size_t k = 0; k < joints.size(); ++k) {
                uint32_t& la = last[joints[k].first];
                uint32_t& lb = last[joints[k].second];
                uint32_t l = std::max(la, lb);
                while (l < levels.size() && levels[l].size() >= width) ++l;
                if (l >= levels.size()) levels.resize(l + 1);
                levels[l].push_back({ids[k], it});
                la = lb = l + 1;
            }
        for (const auto& j : joints) last[j.first] = last[j.second] = 0;
        for (const auto& l : levels) {
            for (const auto& e : l) {
                entry.push_back(e.first);
                iteration.push_back(e.second);
            }
            level_start.push_back((uint32_t)entry.size());
        }
        group_level.push_back((uint32_t)level_start.size() - 1);
    }
};

}  // namespace bg
