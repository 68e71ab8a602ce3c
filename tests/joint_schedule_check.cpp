// Checks of JointSchedule (blobs_amd/csrc/joint_schedule.hpp) on the CPU, run by
// test_joint_schedule.py: `random` against the definition, solve by solve;
// `mesh SIDE ITERATIONS` prints the seconds that one wide component takes.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "joint_schedule.hpp"

using Joints = std::vector<std::pair<uint32_t, uint32_t>>;

// The first level after those of the solve's bodies that has room, searched one by one.
static bool same_as_definition(const Joints& joints, uint32_t bodies, uint32_t iterations, uint32_t width) {
    std::vector<uint32_t> ids(joints.size()), last(bodies, 0), after(bodies, 0);
    for (size_t k = 0; k < ids.size(); ++k) ids[k] = 1000u + (uint32_t)k;
    bg::JointSchedule s;
    s.add_group(joints, ids, iterations, last, width);
    s.add_group(joints, ids, iterations, last, width);
    std::vector<std::vector<std::pair<uint32_t, uint32_t>>> levels;
    for (uint32_t it = 0; it < iterations; ++it)
        for (size_t k = 0; k < joints.size(); ++k) {
            uint32_t l = std::max(after[joints[k].first], after[joints[k].second]);
            while (l < levels.size() && levels[l].size() >= width) ++l;
            if (l >= levels.size()) levels.resize(l + 1);
            levels[l].push_back({ids[k], it});
            after[joints[k].first] = after[joints[k].second] = l + 1;
        }
    if (s.groups() != 2 || s.group_level[2] != 2 * levels.size()) return false;
    for (uint32_t v : last)
        if (v != 0) return false;
    for (int g = 0; g < 2; ++g)
        for (size_t l = 0; l < levels.size(); ++l) {
            const uint32_t a = s.level_start[g * levels.size() + l], b = s.level_start[g * levels.size() + l + 1];
            if (b - a != levels[l].size()) return false;
            for (uint32_t e = a; e < b; ++e)
                if (s.entry[e] != levels[l][e - a].first || s.iteration[e] != levels[l][e - a].second) return false;
        }
    return true;
}

int main(int argc, char** argv) {
    if (argc > 3 && !strcmp(argv[1], "mesh")) {
        const uint32_t side = (uint32_t)atoi(argv[2]), iterations = (uint32_t)atoi(argv[3]);
        Joints joints;
        for (uint32_t odd = 0; odd < 2; ++odd)  // joints that share no body in a row, so that levels fill up
            for (uint32_t y = 0; y < side; ++y)
                for (uint32_t x = odd; x + 1 < side; x += 2) joints.push_back({y * side + x, y * side + x + 1});
        for (uint32_t odd = 0; odd < 2; ++odd)
            for (uint32_t y = odd; y + 1 < side; y += 2)
                for (uint32_t x = 0; x < side; ++x) joints.push_back({y * side + x, (y + 1) * side + x});
        std::vector<uint32_t> ids(joints.size()), last(side * side, 0);
        for (size_t k = 0; k < ids.size(); ++k) ids[k] = (uint32_t)k;
        bg::JointSchedule s;
        const auto t = std::chrono::steady_clock::now();
        s.add_group(joints, ids, iterations, last, 64);
        printf("%zu %f\n", s.entry.size(), std::chrono::duration<double>(std::chrono::steady_clock::now() - t).count());
        return 0;
    }
    std::mt19937 rng(5);
    for (int k = 0; k < 400; ++k) {
        const uint32_t bodies = 1u + rng() % 60u, n = rng() % 200u, iterations = rng() % 6u, width = 1u + rng() % 9u;
        Joints joints;
        for (uint32_t j = 0; j < n; ++j) joints.push_back({rng() % bodies, rng() % bodies});
        if (!same_as_definition(joints, bodies, iterations, width)) {
            printf("case %d differs\n", k);
            return 1;
        }
    }
    printf("ok\n");
    return 0;
}
