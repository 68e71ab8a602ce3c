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
        std::vector<uint32_t> filled;  // solves of each level
        std::vector<uint32_t> room;    // of each level: itself, or where to look on for one with room
        std::vector<uint32_t> at;      // each solve's level, in the order of the sweep
        at.reserve(joints.size() * iterations);
        for (uint32_t it = 0; it < iterations; ++it)
            for (const auto& j : joints) {
                uint32_t& la = last[j.first];
                uint32_t& lb = last[j.second];
                uint32_t l = std::max(la, lb);
                while (l < room.size() && room[l] != l) {  // (halving the path, or a wide component walks all its levels)
                    if (room[l] < room.size()) room[l] = room[room[l]];
                    l = room[l];
                }
                for (; l >= room.size(); filled.push_back(0)) room.push_back((uint32_t)room.size());
                if (++filled[l] == width) room[l] = l + 1;
                at.push_back(l);
                la = lb = l + 1;
            }
        for (const auto& j : joints) last[j.first] = last[j.second] = 0;
        const size_t first = entry.size();
        std::vector<uint32_t> next(filled.size());
        for (size_t l = 0, n = first; l < filled.size(); ++l) {
            next[l] = (uint32_t)n;
            n += filled[l];
            level_start.push_back((uint32_t)n);
        }
        entry.resize(first + at.size());
        iteration.resize(first + at.size());
        for (size_t s = 0; s < at.size(); ++s) {
            const uint32_t to = next[at[s]]++;
            entry[to] = ids[s % joints.size()];
            iteration[to] = (uint32_t)(s / joints.size());
        }
        group_level.push_back((uint32_t)level_start.size() - 1);
    }
};

}  // namespace bg
