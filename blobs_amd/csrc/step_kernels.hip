// step_kernels.hip -- gfx950 kernels of one `Physics::step` substep.
//
// Reference stage order per substep (physics.rs:401-421): gravity, springs,
// contacts, fixed joints, Verlet update (+ collider transforms), circle
// constraints.  Two device paths implement it:
//
//  * general path (any world), per substep: k_keys_forces (the rebuild's
//    key pass beside gravity + springs per body), the scan and k_cell_scatter
//    (counting sort of the colliders by cell), k_contact_lists (a wave's
//    queue of pairs) and k_contact_merge (per body; k_contacts for the bodies whose lists
//    overflowed), the ordered push-out pass (ordered_contacts.hip), k_joints
//    (a workgroup a group of components, by levels), k_integrate (Verlet, joint
//    rotations, collider transforms, constraints, per body);
//  * fused sphere path (one collider per body, no springs/joints): all stages
//    in one kernel per substep over bodies kept in broadphase-cell order
//    (sphere_kernels.hip).
//
// Contacts are order-independent until a push-out because the reference
// tests the collider snapshot written by the previous Verlet (physics.rs:264,
// 360-366), so the pair set and every correction vector depend only on the
// snapshot; only the summation order on a body position matters, and each
// body sums its own corrections in the reference's (i, j<i) lexicographic
// order.
#include <float.h>

#include "common.hpp"
#include "device_state.hpp"
#include "lds_grid.hpp"
#include "sort.hpp"
#include "step_common.hpp"

namespace bg {

namespace {

constexpr uint32_t kContactThreads = 64;  // block size of k_contacts (block_contacts: one slot per 64 bodies)


// Clips a box of more cells than the table has to the centroid +- 3 sigma of 256 colliders, so
// that the few that flew off (clamped into border cells) do not coarsen the cells of the rest.  Every
// wave works it out for itself, all its lanes, from the same snapshots in the same order: the
// loads hit the cache, and a statistics pass or a barrier would cost more.  294,249 colliders over
// their first 112 steps, as the box grows from 776 to 12,000 units: k_contact_lists 28.0 -> 16.8 us,
// k_keys_forces, this included, 20.4 -> 17.6.
//
// What lies outside may be a group, and crowd a border cell where each of its colliders walks all of
// it: a step of 147,000 colliders with 7% of them 5,000 units off took 12,457 us, against 1,030 with the
// whole box.  So a border cell of more than kBorderCrowd (128 to walk take a wave some 11 us) keeps
// the box whole for kClipHold substeps (one crowded one in 1,024 is about 1%), and so does an upload for
// kClipWait.  A scene that flies apart on all sides comes to that now and then: eight steps of 65,536
// bodies, over their first 200, 8.39 ms, 8.02 with no limit, 8.20 at 256 -- where groups of 3% and 7% to
// one side took up to 18% more than with the whole box -- and 8.63 at 21.
constexpr uint32_t kBorderCrowd = 128, kClipHold = 1024;  // (kClipWait: device_state.hpp)
__device__ __forceinline__ void clip_box(uint32_t (&bb)[4], const KeysArgs& k) {
    constexpr uint32_t kSample = 4;  // a lane
    const float minx = ord2f(bb[0]), miny = ord2f(bb[1]), ex = ord2f(bb[2]) - minx, ey = ord2f(bb[3]) - miny;
    if (k.accum->clip_hold != 0u || k.nc < 16u * kSample * BG_WAVE || !finitef(ex) || !finitef(ey) ||
        !((ex / k.cell + 1.0f) * (ey / k.cell + 1.0f) > (float)k.cells_cap))
        return;
    const uint32_t lane = threadIdx.x & (BG_WAVE - 1), stride = k.nc / (kSample * BG_WAVE);
    float2 x[kSample];
#pragma unroll
    for (uint32_t j = 0; j < kSample; ++j) x[j] = k.xy[(j * BG_WAVE + lane) * stride];
    const float cx = minx + 0.5f * ex, cy = miny + 0.5f * ey;
    float s[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (uint32_t j = 0; j < kSample; ++j) {
        const float dx = x[j].x - cx, dy = x[j].y - cy;
        if (!finitef(dx) || !finitef(dy)) continue;
        s[0] += 1.0f;
        s[1] += dx;
        s[2] += dy;
        s[3] += dx * dx;
        s[4] += dy * dy;
    }
#pragma unroll
    for (int q = 0; q < 5; ++q)
        s[q] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
            (int)wave_prefix(__float_as_uint(s[q]), 0u, AddF32()), BG_WAVE - 1));
    const float mx = s[1] / s[0], my = s[2] / s[0], mg = 2.0f * k.cell;
    const float rx = 3.0f * sqrtf(fmaxf(s[3] / s[0] - mx * mx, 0.0f)) + mg;
    const float ry = 3.0f * sqrtf(fmaxf(s[4] / s[0] - my * my, 0.0f)) + mg;
    if (!finitef(mx) || !finitef(my) || !finitef(rx) || !finitef(ry)) return;
    bb[0] = max(bb[0], f2ord(cx + mx - rx));
    bb[1] = max(bb[1], f2ord(cy + my - ry));
    bb[2] = min(bb[2], f2ord(cx + mx + rx));
    bb[3] = min(bb[3], f2ord(cy + my + ry));
    if (bb[0] > bb[2]) bb[0] = bb[2];
    if (bb[1] > bb[3]) bb[1] = bb[3];
}

// Cell key of collider i's snapshot on the grid fitted to the bounding box
// accumulated since the previous rebuild, and its rank among its cell's
// colliders (counting sort; order inside a cell is arbitrary, no result
// depends on it).  Thread 0 stores the grid and clears the box the coming
// substep accumulates.
template <bool CLIP>
__device__ __forceinline__ void rebuild_key_at(uint32_t i, const KeysArgs& k) {
    const uint32_t* box = k.accum->bbox[k.parity];
    uint32_t bb[4] = {box[0], box[1], box[2], box[3]};
    if (CLIP) clip_box(bb, k);
    const GridParams g = grid_from_bbox(bb, k.cell, k.cells_cap);
    if (i == 0) {
        *k.grid_out = g;
        k.accum->bbox[k.parity ^ 1][0] = 0xFFFFFFFFu;
        k.accum->bbox[k.parity ^ 1][1] = 0xFFFFFFFFu;
        k.accum->bbox[k.parity ^ 1][2] = 0u;
        k.accum->bbox[k.parity ^ 1][3] = 0u;
        k.accum->n_outliers = 0u;
    }
    if (i < k.nc) {
        const float2 x = k.xy[i];
        int32_t cx = cell_coord(x.x, g.ox, g.inv_cell, g.nx);
        int32_t cy = cell_coord(x.y, g.oy, g.inv_cell, g.ny);
        const uint32_t kk = (uint32_t)cy * (uint32_t)g.nx + (uint32_t)cx;
        k.keys[i] = kk;
        k.rank[i] = atomicAdd(&k.cnt[kk], 1u);
    }
}

// Collider i into cell order: slot = cell_start[key] + rank (cell_start is the exclusive scan of
// the counts).  Beside the collider index, each slot gets the record the contact pass tests
// (position, radius, parent body), so a candidate is one load from a cell run.
struct CellScatter {
    const uint32_t* keys;
    const uint32_t* rank;
    uint32_t nc;
    const uint32_t* cell_start;
    uint32_t* vals;
    const float2* abs;
    const float* radius;
    const int32_t* parent;
    float4* rec;
};
__device__ __forceinline__ void scatter_at(uint32_t i, const CellScatter& k) {
    if (i >= k.nc) return;
    const uint32_t slot = k.cell_start[k.keys[i]] + k.rank[i];
    if (slot < k.nc) {  // consistent counts and scan never fail this
        k.vals[slot] = i;
        const float2 x = k.abs[i];
        k.rec[slot] = make_float4(x.x, x.y, k.radius[i], __int_as_float(k.parent[i]));
    }
}
CellScatter cell_scatter_of(const DeviceWorld& d) {
    return {d.keys, d.vals_tmp, d.nc, d.cell_start, d.vals, d.c.abs, d.c.radius, d.c.parent, d.crec};
}

// The counts are cleared for the next rebuild; a crowded border cell is noted for clip_box.
__global__ __launch_bounds__(kThreads) void k_cell_scatter(CellScatter k, uint32_t* cnt, uint32_t n_cnt,
                                                           const GridParams* __restrict__ grid, StepAccum* accum) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    // only the grid's cells were counted (and scanned): clear those
    const uint32_t n_used = grid->ncells + 1u < n_cnt ? grid->ncells + 1u : n_cnt;
    for (uint32_t c = i; c < n_used; c += gridDim.x * blockDim.x) cnt[c] = 0u;
    if (i == 0 && accum->clip_hold != 0u) atomicSub(&accum->clip_hold, 1u);  // (read by the key pass only)
    if (i < k.nc && k.rank[i] >= kBorderCrowd) {
        const uint32_t nx = (uint32_t)grid->nx, cy = k.keys[i] / nx, cx = k.keys[i] - cy * nx;
        if (cx == 0u || cx == nx - 1u || cy == 0u || cy == (uint32_t)grid->ny - 1u)
            atomic_max_if_greater(&accum->clip_hold, kClipHold);
    }
    scatter_at(i, k);
}

// ============================================================ general path

// Gravity + springs -> acc of body b (physics.rs:404-408, springs.rs:25-47).
// A chain of loads: a body's springs are records of their own, in a row, so that only
// the other body's state depends on them (beside the key pass 20.9 us at 65,536
// bodies and 32,768 springs; 23.5 through a list of springs).
__device__ __forceinline__ void forces_at(uint32_t b, const DeviceWorld& d, const SubstepArgs& a) {
    if (b >= d.nb) return;
    uint32_t fl = d.b.bflags[b];
    if (fl & BF_STATIC) return;
    float2 acc = a.fresh ? d.b.acc[b] : make_float2(0.0f, 0.0f);
    float gm = d.b.gmod[b];
    acc.x = acc.x + a.gx * gm;
    acc.y = acc.y + a.gy * gm;
    const float m = d.b.mass[b];
    const uint32_t k1 = d.bs_start[b + 1];
    uint32_t k = d.bs_start[b];
    if (k < k1) {
        // each record and the other body's state load while the spring before is worked out
        const float2 own_p = d.b.pos[b], own_v = d.b.vel[b];
        float4 rec = d.bs_rec[k], next = d.bs_rec[min(k + 1u, k1 - 1u)];
        uint32_t o = __float_as_uint(rec.x) & 0x7FFFFFFFu;
        float2 op = d.b.pos[o], ov = d.b.vel[o];
        for (; k < k1; ++k) {
            const bool is_b = (__float_as_uint(rec.x) >> 31) != 0u;
            const float2 pa = is_b ? op : own_p, pb = is_b ? own_p : op;
            const float2 va = is_b ? ov : own_v, vb = is_b ? own_v : ov;
            const float rest = rec.y, stiff = rec.z, damp = rec.w;
            rec = next;
            o = __float_as_uint(rec.x) & 0x7FFFFFFFu;
            next = d.bs_rec[min(k + 2u, k1 - 1u)];
            op = d.b.pos[o];
            ov = d.b.vel[o];
            float dx = pb.x - pa.x, dy = pb.y - pa.y;
            float dist = vlen(dx, dy);
            float ux = dx / dist, uy = dy / dist;
            float rvx = va.x - vb.x, rvy = va.y - vb.y;
            float dot = rvx * ux + rvy * uy;
            float cd = damp * dot;
            float dfx = cd * ux, dfy = cd * uy;
            float mag = stiff * (dist - rest);
            float fx = ux * (mag - dfx), fy = uy * (mag - dfy);
            acc.x = acc.x + (is_b ? -fx : fx) / m;
            acc.y = acc.y + (is_b ? -fy : fy) / m;
        }
    }
    d.b.acc[b] = acc;
}

// The substep's first launch on the general path: the collider keys of the
// rebuild (blocks [0, key_blocks), when the substep rebuilds) and gravity +
// springs (the rest).  The two are independent: keys read the collider
// snapshots, forces the body positions and velocities.
__global__ __launch_bounds__(kThreads) void k_keys_forces(KeysArgs k, uint32_t key_blocks, DeviceWorld d,
                                                         SubstepArgs a) {
    if (blockIdx.x < key_blocks) {
        rebuild_key_at<true>(blockIdx.x * blockDim.x + threadIdx.x, k);
    } else if (a.has_springs) {
        forces_at((blockIdx.x - key_blocks) * blockDim.x + threadIdx.x, d, a);
    }
}

constexpr uint32_t kColStage = 8;  // colliders per body staged in LDS by k_contacts

// Contacts (physics.rs:241-317), one thread per body over its colliders, in
// blocks of kContactThreads.  With `list`, only the bodies listed there (count
// in cfb_n[0], grid-stride) and without counting or events: the bodies whose
// collider lists overflowed in k_contact_lists, which counted their contacts.
template <bool GROUPS, bool SENSORS>
__global__ __launch_bounds__(kContactThreads) void k_contacts(DeviceWorld d, SubstepArgs a, const uint32_t* list) {
    // the body's first kColStage colliders (x, y, radius, index), loaded together up front
    // so that the walk over its colliders does not wait on two dependent loads per collider
    __shared__ float4 s_col[kColStage][kContactThreads];
    uint32_t all_count = 0, all_flags = 0;
    const uint32_t lane = threadIdx.x;
    const uint32_t n_items = list ? d.cfb_n[0] : d.nb;
    const uint32_t stride = list ? gridDim.x * blockDim.x : n_items;  // without a list: one body per thread
    for (uint32_t item = blockIdx.x * blockDim.x + threadIdx.x; item < n_items; item += stride) {
        const uint32_t b = list ? list[item] : item;
        const GridParams g = *d.grid;
        float2 p = d.b.pos[b];
        d.pos_pre[b] = p;  // the ordered pass re-sums from here if a push-out happens
        const float mown = d.b.mass[b];
        ContactList<16, uint64_t> L;
        L.init();
        const uint32_t k0 = d.bc_start[b], k1 = d.bc_start[b + 1];
        if (k1 > k0) {
            // an index past the end repeats the last collider (same slot, same values)
            uint32_t cc[kColStage];
#pragma unroll
            for (uint32_t u = 0; u < kColStage; ++u) cc[u] = d.bc_list[min(k0 + u, k1 - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < kColStage; ++u) {
                const float2 x = d.c.abs[cc[u]];
                s_col[min(u, k1 - k0 - 1u)][lane] = make_float4(x.x, x.y, d.c.radius[cc[u]], __uint_as_float(cc[u]));
            }
        }
        // one enumeration of this body's contact corrections, in visit order
        auto enumerate = [&](auto&& emit) {
            for (uint32_t kk = k0; kk < k1; ++kk) {
                uint32_t c;
                float2 xa;
                float ra;
                if (kk - k0 < kColStage) {
                    const float4 sc = s_col[kk - k0][lane];
                    c = __float_as_uint(sc.w);
                    xa = make_float2(sc.x, sc.y);
                    ra = sc.z;
                } else {
                    c = d.bc_list[kk];
                    xa = d.c.abs[c];
                    ra = d.c.radius[c];
                }
                if (!finitef(xa.x) || !finitef(xa.y)) continue;
                uint2 ga = make_uint2(0, 0);
                if (GROUPS) ga = d.c.groups[c];
                const bool sen_a = SENSORS ? (d.c.cflags[c] & 1u) : false;
                const float Q = ra + a.rmax;
                scan_stencil(g, d.cell_start, d.nc, d.crec, xa.x - a.drift_prev_x, xa.y - a.drift_prev_y, Q,
                             [&](uint32_t t, const float4 (&rb)[4], uint32_t nv) {
                    // slot records (the sort ran on this substep's positions); the collider
                    // itself and its body's other colliders share the parent b.  All four
                    // are tested first, then the hits' collider indices and partner masses
                    // are loaded together, then the hits are taken in slot order.
                    // axis = A - B with A the higher collider index; b - a == -(a - b) up to
                    // the sign of a zero, so the unoriented difference decides and the axis
                    // is formed for a hit only
                    bool hit[4];
                    float dx[4], dy[4], dot[4], rs[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) {
                        const int32_t pj = __float_as_int(rb[u].w);
                        dx[u] = xa.x - rb[u].x;
                        dy[u] = xa.y - rb[u].y;
                        rs[u] = ra + rb[u].z;
                        dot[u] = dx[u] * dx[u] + dy[u] * dy[u];
                        hit[u] = u < nv && pj >= 0 && pj != (int32_t)b &&
                                 !(dot[u] > (rs[u] * rs[u]) * 1.00000095367431640625f) && sqrt_lt(dot[u], rs[u]);
                    }
                    uint32_t jj[4];
                    float mp[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) {
                        jj[u] = 0u;
                        mp[u] = 0.0f;
                        if (hit[u]) {
                            jj[u] = d.vals[t + u];
                            mp[u] = d.b.mass[__float_as_int(rb[u].w)];
                        }
                    }
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) {
                        if (!hit[u]) continue;
                        const uint32_t j = jj[u];
                        if (GROUPS) {
                            uint2 gb = d.c.groups[j];
                            if (!((ga.x & gb.y) != 0u && (gb.x & ga.y) != 0u)) continue;
                        }
                        const bool isA = c > j;
                        const float ax = isA ? dx[u] : rb[u].x - xa.x, ay = isA ? dy[u] : rb[u].y - xa.y;
                        const uint64_t key = isA ? (((uint64_t)c << 32) | j) : (((uint64_t)j << 32) | c);
                        emit(key, isA, j, __float_as_int(rb[u].w), ax, ay, sqrtf(dot[u]), rs[u], sen_a, mp[u]);
                    }
                });
            }
        };
        uint32_t count = 0, flags = 0;
        // Correction vector of one contact for this body's side.  A pair whose
        // snapshots coincide takes the push-out branch (physics.rs:272-286), which
        // makes the rest of the pass order dependent: its row (the A collider) is
        // recorded once for k_contacts_ordered, which replays the affected pairs in
        // reference order and rewrites the positions they touch.  The value summed
        // here for such a pair is a placeholder.
        auto correction = [&](bool first, auto&& sink, uint64_t key, bool isA, uint32_t j, float mpart, float ax,
                              float ay, float dist, float rs, bool sen_a) {
            float px = 0.0f, py = 0.0f;
            const bool pushed = dist < 1e-6f;
            if (pushed) {
                ax = ax + 0.02f;
                dist = vlen(ax, ay);
                px = isA ? 0.01f : -0.01f;
                py = isA ? 0.0f : -0.0f;
                if (first) {
                    flags |= INFO_PUSH_OUT;
                    if (isA) {
                        const uint32_t row = (uint32_t)(key >> 32), bit = 1u << (row & 31u);
                        if (!(atomicOr(&d.ord_mark[row >> 5], bit) & bit)) d.ord_rows[atomicAdd(d.ord_n, 1u)] = row;
                    }
                }
            }
            const bool sen_b = SENSORS ? (d.c.cflags[j] & 1u) : false;
            if (sen_a || sen_b) {
                if (pushed) sink(key, px, py);
                return;
            }
            const float mA = isA ? mown : mpart, mB = isA ? mpart : mown;
            const float ratio = 1.0f - mA / (mA + mB);
            const float nx = ax / dist, ny = ay / dist;
            if (first && (nx != nx || ny != ny)) flags |= ERR_NAN_NORMAL;
            const float delta = rs - dist;
            float cx, cy;
            if (isA) {
                const float k = ratio * delta;
                cx = k * nx;
                cy = k * ny;
            } else {
                const float k = (1.0f - ratio) * delta;
                cx = -(k * nx);
                cy = -(k * ny);
            }
            if (pushed) {
                cx = px + cx;
                cy = py + cy;
            }
            sink(key, cx, cy);
        };
        enumerate([&](uint64_t key, bool isA, uint32_t j, int32_t pj, float ax, float ay, float dist, float rs,
                      bool sen_a, float mp) {
            if (isA && !list) ++count;
            correction(true, [&](uint64_t k, float x, float y) { L.add(k, x, y); }, key, isA, j, mp, ax, ay, dist,
                       rs, sen_a);
        });
        if (d.events && count > 0) {
            // collision events of the pairs whose A collider is this body's (physics.rs:288-311);
            // velocities are the bodies' calculated_velocity before the contact pass
            unsigned long long e = atomicAdd(&d.accum->event_count, (unsigned long long)count);
            const float2 va = d.b.vel[b];
            enumerate([&](uint64_t key, bool isA, uint32_t j, int32_t pj, float ax, float ay, float dist, float rs,
                          bool sen_a, float) {
                if (!isA) return;
                if (e < d.event_cap) {
                    DevEvent ev;
                    ev.sub = a.sub_global;
                    ev.a = (uint32_t)(key >> 32);
                    ev.b = (uint32_t)key;
                    ev.pad = 0;
                    ev.va = va;
                    ev.vb = d.b.vel[pj];
                    d.events[e] = ev;
                }
                ++e;
            });
        }
        if (L.n > 0) {
            const uint32_t total = L.n;
            uint64_t last = L.apply(p);
            uint32_t done = total < 16 ? total : 16;
            // more corrections than the register list holds: each further pass over
            // the candidates collects the 16 smallest keys above the last one applied
            // and applies them, so the order stays ascending
            while (done < total) {
                L.init();
                enumerate([&](uint64_t key, bool isA, uint32_t j, int32_t pj, float ax, float ay, float dist,
                              float rs, bool sen_a, float mp) {
                    correction(
                        false,
                        [&](uint64_t k, float x, float y) {
                            if (k > last) L.add(k, x, y);
                        },
                        key, isA, j, mp, ax, ay, dist, rs, sen_a);
                });
                if (L.n == 0) break;
                last = L.apply(p);
                done += L.n < 16 ? L.n : 16;
            }
            d.b.pos[b] = p;
        }
        all_count += count;
        all_flags |= flags;
    }
    // (a block is one wave; contacts go to its slot, summed on the host when queried)
    if (all_flags) atomicOr(&d.accum->error_flags, all_flags);
    const uint32_t sum = wave_sum_u32(all_count);
    if (lane == 0 && sum) d.block_contacts[blockIdx.x] += sum;
}

constexpr uint32_t kColList = 16;   // corrections a collider keeps (the smallest keys)
constexpr uint32_t kPairCap = 320;  // pairs a wave queues
constexpr int kDirectRegs = 4;      // corrections of a collider outside the queue sorted in registers

// Contacts, first half of the two-kernel form: every collider walks its own
// stencil (physics.rs:248-300 for the pairs it is in), counts the pairs it is
// A in, sends their events, records push-out rows, and keeps its body's side
// of each correction -- the kColList smallest keys, in key order -- in
// clist[i * nc + c], with the full count in ccnt[c].
//
// Bound by the chain of dependent loads (cell table, records, partners) and
// by corrections that few lanes of a wave run at a time: hits are few (0.04 to
// 0.6 a collider of the scene of 294,249), candidates about five.  So a thread
// marks the candidates of its collider within reach, the wave queues the marked pairs,
// works them out a pair a lane whoever's they are, and each thread then takes
// its own in ascending partner: 36.4 us over the scene's first 112 steps, against 48.1 with a
// thread doing all of its collider's contacts, sixteen sorted in registers (166
// registers, three waves a SIMD); 6.2 against 14.2 at 1,115 colliders.
struct ListsLds {
    float4 own[BG_WAVE];     // (x, y, radius, body's mass)
    uint2 id[BG_WAVE];       // collider, body
    uint2 pair[kPairCap];    // own lane, partner's slot; then (partner, -) or (kNil, -)
    float2 res[kPairCap];
};
// One wave's LDS accesses keep their order; the compiler has to as well.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ uint64_t merge_key(float4 v) {
    return ((uint64_t)__float_as_uint(v.x) << 32) | __float_as_uint(v.y);
}

template <bool GROUPS, bool SENSORS>
__device__ __forceinline__ void contact_lists(const DeviceWorld& d, const SubstepArgs& a, ListsLds& lds, uint32_t slot,
                                              uint32_t count_slot) {
    // threads walk the colliders in cell order (the order the key pass just sorted them
    // into): a wave's colliders are neighbours, so their candidate records overlap in cache
    // (an XCD takes a contiguous range of them), and each one's own record is the slot's
    // (x, y, radius, parent), loaded coalesced
    float4* s_own = lds.own;
    uint2 *s_id = lds.id, *s_pair = lds.pair;
    float2* s_res = lds.res;
    const uint32_t lane = threadIdx.x & (BG_WAVE - 1);
    if (slot == 0) d.cfb_n[0] = 0u;  // k_contact_merge fills the fallback list after this
    uint32_t count = 0, flags = 0;
    uint32_t c = 0, n = 0, first = 0, n_put = 0;
    bool direct = false;
    int32_t b = -1;
    float4 own = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (slot < d.nc) {
        c = d.vals[slot];
        own = d.crec[slot];
        b = __float_as_int(own.w);
        if (!finitef(own.x) || !finitef(own.y)) b = -1;
    }
    // One pair from the side of collider `cc` (o: its position, radius and mass) with the candidate
    // record rb, collider j, mass mp: put(x, y) with the correction, if it is a contact that has
    // one.  axis = A - B with A the higher collider index; b - a == -(a - b) up to the sign of a
    // zero, so the unoriented difference decides.  A push-out only records its row (as k_contacts).
    auto contact = [&](uint32_t cc, int32_t body, const float4& o, const float4& rb, uint32_t j, float mp,
                       auto&& put) {
        float ax = o.x - rb.x, ay = o.y - rb.y;
        const float rs = o.z + rb.z;
        const float dot = ax * ax + ay * ay;
        if (dot > (rs * rs) * 1.00000095367431640625f) return;
        float dist = sqrtf(dot);
        if (!(dist < rs)) return;
        if (GROUPS) {
            const uint2 ga = d.c.groups[cc], gb = d.c.groups[j];
            if (!((ga.x & gb.y) != 0u && (gb.x & ga.y) != 0u)) return;
        }
        const bool isA = cc > j;
        if (isA) {
            ++count;
            if (d.events) {  // physics.rs:288-311
                const unsigned long long e = atomicAdd(&d.accum->event_count, 1ull);
                if (e < d.event_cap) {
                    DevEvent ev;
                    ev.sub = a.sub_global;
                    ev.a = cc;
                    ev.b = j;
                    ev.pad = 0;
                    ev.va = d.b.vel[body];
                    ev.vb = d.b.vel[__float_as_int(rb.w)];
                    d.events[e] = ev;
                }
            }
        }
        ax = isA ? ax : rb.x - o.x;
        ay = isA ? ay : rb.y - o.y;
        float px = 0.0f, py = 0.0f;
        const bool pushed = dist < 1e-6f;
        if (pushed) {
            ax = ax + 0.02f;
            dist = vlen(ax, ay);
            px = isA ? 0.01f : -0.01f;
            py = isA ? 0.0f : -0.0f;
            flags |= INFO_PUSH_OUT;
            if (isA) {
                const uint32_t bit = 1u << (cc & 31u);
                if (!(atomicOr(&d.ord_mark[cc >> 5], bit) & bit)) d.ord_rows[atomicAdd(d.ord_n, 1u)] = cc;
            }
        }
        if (SENSORS && ((d.c.cflags[cc] | d.c.cflags[j]) & 1u)) {
            if (pushed) put(px, py);
            return;
        }
        const float mA = isA ? o.w : mp, mB = isA ? mp : o.w;
        const float ratio = 1.0f - mA / (mA + mB);
        const float nx = ax / dist, ny = ay / dist;
        if (nx != nx || ny != ny) flags |= ERR_NAN_NORMAL;
        const float delta = rs - dist;
        const float k = isA ? ratio * delta : (1.0f - ratio) * delta;
        float cx = isA ? k * nx : -(k * nx), cy = isA ? k * ny : -(k * ny);
        if (pushed) {
            cx = px + cx;
            cy = py + cy;
        }
        put(cx, cy);
    };
    auto store = [&](uint32_t row, uint32_t j, float x, float y) {
        if (row < kColList)
            d.clist[(size_t)row * d.nc + c] =
                make_float4(__uint_as_float(max(c, j)), __uint_as_float(min(c, j)), x, y);
    };

    // ---- mark
    LdsRect cells = {0, 0, 0, 0};
    LdsRows rows = {0, 0, 0, 0, 0, 0, false};
    uint64_t marked = 0;
    const uint32_t nx = (uint32_t)d.grid->nx;
    auto near = [&](const float4& rb) {
        const float dx = own.x - rb.x, dy = own.y - rb.y, rs = own.z + rb.z;
        const int32_t pj = __float_as_int(rb.w);
        // (the collider itself and its body's other colliders share the parent b)
        return (pj >= 0) & (pj != b) & !(dx * dx + dy * dy > (rs * rs) * 1.00000095367431640625f);
    };
    if (b >= 0) {
        const GridParams g = *d.grid;
        const float2 q = make_float2(own.x - a.drift_prev_x, own.y - a.drift_prev_y);
        const float R = stencil_reach(q, own.z + a.rmax);
        own.w = d.b.mass[b];
        cells.cx1 = g.nx - 1;
        cells.cy1 = g.ny - 1;
        if (R < 1e30f && finitef(q.x) && finitef(q.y)) {
            cells.cx0 = cell_coord(q.x - R, g.ox, g.inv_cell, g.nx);
            cells.cx1 = cell_coord(q.x + R, g.ox, g.inv_cell, g.nx);
            cells.cy0 = cell_coord(q.y - R, g.oy, g.inv_cell, g.ny);
            cells.cy1 = cell_coord(q.y + R, g.oy, g.inv_cell, g.ny);
        }
        rows = flat_rows(d.cell_start, nx, cells);
        static_assert(kLdsFlat <= 64, "one mask");
        direct = !rows.flat;
        const uint32_t n_flat = rows.n;
        for (uint32_t f = 0; f < n_flat; f += 4) {
            float4 rb[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) rb[u] = d.crec[min(rows.slot(min(f + u, n_flat - 1u)), d.nc - 1u)];
            uint32_t bits = 0;
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) bits |= (f + u < n_flat) && near(rb[u]) ? 1u << u : 0u;
            marked |= (uint64_t)bits << f;
        }
    }
    s_own[lane] = own;
    s_id[lane] = make_uint2(c, (uint32_t)b);
    n = (uint32_t)__popcll(marked);
    const uint32_t incl = wave_prefix(n, 0u, AddU32());
    first = incl - n;
    const bool fits = incl <= kPairCap;  // (true up to some lane)
    const uint64_t fit_lanes = __ballot(fits);
    const uint32_t queued =
        fit_lanes ? (uint32_t)__builtin_amdgcn_readlane((int)incl, 63 - __builtin_clzll(fit_lanes)) : 0u;
    if (!fits && n > 0) {
        direct = true;
        n = 0;
    }
    if (fits)
        for (uint32_t e = first; marked != 0; ++e, marked &= marked - 1)
            s_pair[e] = make_uint2(lane, rows.slot((uint32_t)__builtin_ctzll(marked)));
    wave_sync();
    // ---- correct: a pair a lane
    for (uint32_t e = lane; e < queued; e += BG_WAVE) {
        const uint2 pr = s_pair[e];
        const float4 rb = d.crec[pr.y];
        const uint32_t j = d.vals[pr.y];
        const uint2 id = s_id[pr.x];
        s_pair[e].x = kNil;
        contact(id.x, (int32_t)id.y, s_own[pr.x], rb, j, d.b.mass[__float_as_int(rb.w)], [&](float x, float y) {
            s_pair[e].x = j;
            s_res[e] = make_float2(x, y);
        });
    }
    wave_sync();
    // ---- each collider's own, in ascending partner: for this collider c the pair key (max, min) of
    // (c, j) orders as j does (every j < c before every j > c, each side by j)
    for (uint32_t next = 0; n_put < n; ++n_put) {
        uint32_t best = kNil, at = 0;
        for (uint32_t e = first; e < first + n; ++e) {
            const uint32_t j = s_pair[e].x;
            if (j >= next && j < best) {
                best = j;
                at = e;
            }
        }
        if (best == kNil) break;
        store(n_put, best, s_res[at].x, s_res[at].y);
        next = best + 1u;
    }
    if (direct) {  // more candidates than a flat list, or no room in the queue
        // The first few contacts are sorted in registers; all go to the list as they are found, and
        // are sorted there if they are more.  (One large collider sends everyone here: a step of 5,000
        // bodies with one of 12 units 2,747 us, 5,559 with a record a load and a pass for every four
        // contacts; 50,000 bodies 3,646 and 7,246.)
        ContactList<kDirectRegs, uint32_t> L;
        L.init();
        for (int32_t cy = cells.cy0; cy <= cells.cy1; ++cy) {
            const uint32_t row = (uint32_t)cy * nx;
            const uint32_t t1 = min(d.cell_start[row + (uint32_t)cells.cx1 + 1u], d.nc);
            for (uint32_t t = d.cell_start[row + (uint32_t)cells.cx0]; t < t1; t += 4) {
                // (four records load together: a walk of hundreds waits for each of its loads)
                float4 four[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) four[u] = d.crec[min(t + u, t1 - 1u)];
                uint32_t bits = 0;
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) bits |= t + u < t1 && near(four[u]) ? 1u << u : 0u;
                for (; bits != 0; bits &= bits - 1) {
                    const uint32_t slot_b = t + (uint32_t)__builtin_ctz(bits);
                    const float4 rb = d.crec[slot_b];
                    const uint32_t j = d.vals[slot_b];
                    contact(c, b, own, rb, j, d.b.mass[__float_as_int(rb.w)], [&](float x, float y) {
                        store(L.n, j, x, y);
                        L.add(j, x, y);
                    });
                }
            }
        }
        n_put = L.n;
        if (n_put <= (uint32_t)kDirectRegs) {
#pragma unroll
            for (int i = 0; i < kDirectRegs; ++i)
                if ((uint32_t)i < n_put) store((uint32_t)i, L.key[i], L.cx[i], L.cy[i]);
        } else if (n_put <= kColList) {  // (the count alone matters past that)
            float4* list = d.clist + c;
            for (uint32_t i = 0; i + 1 < n_put; ++i) {
                uint32_t least = i;
                uint64_t key = merge_key(list[(size_t)i * d.nc]);
                for (uint32_t k = i + 1; k < n_put; ++k) {
                    const uint64_t other = merge_key(list[(size_t)k * d.nc]);
                    least = other < key ? k : least;
                    key = other < key ? other : key;
                }
                const float4 v = list[(size_t)i * d.nc];
                list[(size_t)i * d.nc] = list[(size_t)least * d.nc];
                list[(size_t)least * d.nc] = v;
            }
        }
    }
    if (slot < d.nc) d.ccnt[c] = n_put;
    if (flags) atomicOr(&d.accum->error_flags, flags);
    const uint32_t sum = wave_sum_u32(count);
    if (lane == 0 && sum) d.block_contacts[count_slot] += sum;
    wave_sync();  // (the wave's next pass writes the same memory)
}

template <bool GROUPS, bool SENSORS>
__global__ __launch_bounds__(kContactThreads) void k_contact_lists(DeviceWorld d, SubstepArgs a) {
    static_assert(kContactThreads == BG_WAVE, "a block is one wave");
    __shared__ ListsLds lds;
    contact_lists<GROUPS, SENSORS>(d, a, lds, xcd_block(blockIdx.x, gridDim.x) * kContactThreads + threadIdx.x,
                                   blockIdx.x);
}

// Second half: adds each body's corrections to its position in key order --
// the reference's (i, j<i) order on this body.  kMergeLanes lanes a body, a
// collider each: a collider's list is in key order, so a step takes the least
// head of the lanes' lists (its keys are the body's alone) and that lane moves
// on.  A body of more colliders is merged by one lane, kMergeRegs keys at a
// time.  A body with a collider past kColList corrections goes to the fallback
// list (k_contacts in list mode re-walks it).
//
// Bound by the chain of loads (colliders, counts, corrections): a lane a
// body, its corrections staged in 1 KB of LDS each, kept two waves a CU and
// took 24.5 us at 65,536 bodies with one to three corrections each; this takes 17.1.
constexpr uint32_t kMergeLanes = 8;
constexpr uint32_t kMergeAhead = 2;  // corrections a lane loads before its count is known
constexpr int kMergeRegs = 6;

// (whole waves: thread t of the pass)
__device__ __forceinline__ void contact_merge(const DeviceWorld& d, uint32_t t) {
    const uint32_t b = t / kMergeLanes, r = t % kMergeLanes;
    uint32_t k0 = 0, k1 = 0;
    float2 p = make_float2(0.0f, 0.0f);
    if (b < d.nb) {
        k0 = d.bc_start[b];
        k1 = d.bc_start[b + 1];
        p = d.b.pos[b];
        if (r == 0) d.pos_pre[b] = p;  // the ordered pass re-sums from here if a push-out happens
    }
    const bool few = k1 - k0 <= kMergeLanes;
    uint32_t c = 0, n = 0;
    float4 ahead[kMergeAhead];
    if (few && r < k1 - k0) {
        c = d.bc_list[k0 + r];
        n = d.ccnt[c];
#pragma unroll
        for (uint32_t i = 0; i < kMergeAhead; ++i) ahead[i] = d.clist[(size_t)i * d.nc + c];
    }
    // the body's lanes: bits of this group in a ballot
    const uint32_t group = (threadIdx.x & (BG_WAVE - 1)) & ~(kMergeLanes - 1);
    auto any_of_group = [&](bool v) { return ((__ballot(v) >> group) & ((1u << kMergeLanes) - 1u)) != 0u; };
    bool fallback = any_of_group(n > kColList);
    if (fallback) n = 0;
    const bool hit = any_of_group(n > 0);
    float4 head = ahead[0];
    uint64_t key = n > 0 ? merge_key(head) : ~0ull;
    for (uint32_t i = 0; __any(key != ~0ull);) {
        uint64_t least = key;
#pragma unroll
        for (uint32_t o = 1; o < kMergeLanes; o *= 2) {
            const uint64_t other = __shfl_xor((unsigned long long)least, o, BG_WAVE);
            least = other < least ? other : least;
        }
        const bool mine = least != ~0ull && key == least;
        const uint64_t who = __ballot(mine);
        const uint32_t in_group = (uint32_t)(who >> group) & ((1u << kMergeLanes) - 1u);
        const uint32_t lane = group + (in_group ? (uint32_t)__builtin_ctz(in_group) : 0u);
        const float cx = __shfl(head.z, (int)lane, BG_WAVE), cy = __shfl(head.w, (int)lane, BG_WAVE);
        if (in_group) {
            p.x = p.x + cx;
            p.y = p.y + cy;
        }
        if (mine) {
            ++i;
            key = ~0ull;
            if (i < n) {
                head = i < kMergeAhead ? ahead[kMergeAhead - 1] : d.clist[(size_t)i * d.nc + c];
                key = merge_key(head);
            }
        }
    }
    static_assert(kMergeAhead == 2, "the two loaded ahead");
    if (b >= d.nb || r != 0) return;
    if (!few) {
        ContactList<kMergeRegs, uint64_t> L;
        uint64_t last = 0;
        for (uint32_t pass = 0;; ++pass) {
            L.init();
            for (uint32_t k = k0; k < k1 && !fallback; ++k) {
                const uint32_t ck = d.bc_list[k], m = d.ccnt[ck];
                fallback |= m > kColList;
                for (uint32_t i = 0; i < m && !fallback; ++i) {
                    const float4 v = d.clist[(size_t)i * d.nc + ck];
                    if (pass == 0 || merge_key(v) > last) L.add(merge_key(v), v.z, v.w);
                }
            }
            if (fallback || L.n == 0) break;
            last = L.apply(p);
            if (L.n <= (uint32_t)kMergeRegs) break;
        }
        if (!fallback) d.b.pos[b] = p;
    } else if (hit) {
        d.b.pos[b] = p;
    }
    if (fallback) d.cfb_list[atomicAdd(d.cfb_n, 1u)] = b;
}

__global__ __launch_bounds__(kThreads) void k_contact_merge(DeviceWorld d) {
    contact_merge(d, blockIdx.x * blockDim.x + threadIdx.x);
}

// Rotation correction of one joint from its axis (physics.rs:462-469): the
// reference adds corr * dt to rotation a and subtracts it from rotation b.
// Positions never read rotations inside the joint stage (anchors are not
// rotated, Q7), so these can be evaluated after the position sweep.
__device__ __forceinline__ float joint_rotation_corr(float dx, float dy, float jtarget) {
    float angle_a = atan2_f32(dy, dx);
    float angle_b = -atan2_f32(dy, -dx);
    float diff = (angle_b - angle_a) - jtarget;
    return diff * 0.5f;
}

// Fixed joints (physics.rs:424-477): a workgroup a group of components
// (components touch disjoint bodies).  Its first wave sweeps the positions
// level by level, a lane a solve (joint_schedule.hpp: the sequential sweep's
// very positions), on LDS copies of the bodies and joint records; the joint's
// mass terms depend on calculated_mass only, so they come in precomputed and
// stay off the chain.  Then all the threads work out the solves' rotation
// steps from the axes, an atan2 pair each, and k_integrate adds them per body
// in the order of the sweep: iterations, then joints in arena order.
//
// Bound by the chain: a level is two LDS reads, a root, two divides and two
// writes, and a lane a component took one such step for each of the largest's
// solves (52, against 24 levels), with two f64 atan2 a solve left to its two
// bodies' threads in a row.  16,384 joints: this kernel and k_integrate took
// 27.6 + 24.6 us a substep that way; a pass of 64 substeps fell from 14.1 to 9.9 ms.
constexpr uint32_t kJointThreads = 256;
constexpr uint32_t kStageJoints = 256, kStageBodies = 384, kStageSolves = 1024, kStageLevels = 512;

struct JointRec {
    float4 anchor, mass;
    float dist;
    uint32_t a, b;  // body list index | static << 31
};

struct JointsLds {
    float4 s_anchor[kStageJoints], s_mass[kStageJoints];
    float2 s_len[kStageJoints];
    uint2 s_ab[kStageJoints];
    float2 s_pos[kStageBodies];
    int32_t s_gid[kStageBodies];
    uint32_t s_level[kStageLevels + 1];
    uint2 s_entry[kStageSolves];
    float2 s_axis[kStageSolves];
};
template <uint32_t NT>
__device__ __forceinline__ void joint_group(const DeviceWorld& d, float h, uint32_t group, JointsLds& lds) {
    auto &s_anchor = lds.s_anchor, &s_mass = lds.s_mass;
    auto& s_len = lds.s_len;
    auto& s_pos = lds.s_pos;
    auto& s_axis = lds.s_axis;
    auto& s_ab = lds.s_ab;
    auto& s_entry = lds.s_entry;
    auto& s_gid = lds.s_gid;
    auto& s_level = lds.s_level;
    const JointGroup g = d.jg[group];
    const uint32_t tid = threadIdx.x, nq = g.q1 - g.q0, nbod = g.b1 - g.b0, nl = g.l1 - g.l0;
    const uint32_t e0 = d.jl_start[g.l0], n = d.jl_start[g.l1] - e0;
    const bool staged = nq <= kStageJoints && nbod <= kStageBodies && nl <= kStageLevels && n <= kStageSolves;
    if (staged) {
        for (uint32_t i = tid; i < nbod; i += NT) {
            const int32_t b = d.jg_body[g.b0 + i];
            s_gid[i] = b;
            s_pos[i] = d.b.pos[b];
        }
        for (uint32_t i = tid; i < nq; i += NT) {
            s_anchor[i] = d.jq_anchor[g.q0 + i];
            s_mass[i] = d.jq_mass[g.q0 + i];
            s_len[i] = d.jq_len[g.q0 + i];
            s_ab[i] = d.jq_ab[g.q0 + i];
        }
        for (uint32_t i = tid; i <= nl; i += NT) s_level[i] = d.jl_start[g.l0 + i] - e0;
        for (uint32_t i = tid; i < n; i += NT) s_entry[i] = d.j_entry[e0 + i];
    }
    __syncthreads();
    uint32_t flags = 0;
    // one solve: axis to `axis`, positions through get and put; body a's write comes first
    auto solve = [&](const JointRec& r, auto&& get, auto&& put) {
        const uint32_t ia = r.a & 0x7FFFFFFFu, ib = r.b & 0x7FFFFFFFu;
        float2 pa = get(ia), pb = get(ib), axis;
        if (joint_positions(pa, pb, make_float2(r.anchor.x, r.anchor.y), make_float2(r.anchor.z, r.anchor.w), r.dist,
                            r.mass, (r.a >> 31) != 0u, (r.b >> 31) != 0u, axis.x, axis.y, flags)) {
            put(ia, pa);
            put(ib, pb);
        }
        return axis;
    };
    if (tid < BG_WAVE) {
        if (staged) {
            // the next level's record loads while the current one works
            uint32_t e = 0, e_next = 0;
            bool have = false, have_next = false;
            JointRec r, r_next;
            auto load = [&](uint32_t l) {
                e_next = s_level[l] + tid;
                have_next = e_next < s_level[l + 1];
                if (!have_next) return;
                const uint32_t q = s_entry[e_next].x;
                r_next.anchor = s_anchor[q];
                r_next.mass = s_mass[q];
                r_next.dist = s_len[q].x;
                const uint2 ab = s_ab[q];
                r_next.a = ab.x;
                r_next.b = ab.y;
            };
            if (nl > 0) load(0);
            for (uint32_t l = 0; l < nl; ++l) {
                e = e_next;
                have = have_next;
                r = r_next;
                if (l + 1 < nl) load(l + 1);
                if (have)
                    s_axis[e] = solve(r, [&](uint32_t i) { return s_pos[i]; },
                                      [&](uint32_t i, float2 p) { s_pos[i] = p; });
                // the next level's lanes read what this one's wrote: one wave's LDS accesses keep
                // their order, the compiler has to as well
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        } else {
            for (uint32_t l = 0; l < nl; ++l) {
                const uint32_t end = d.jl_start[g.l0 + l + 1];
                for (uint32_t e = d.jl_start[g.l0 + l] + tid; e < end; e += BG_WAVE) {
                    const uint2 en = d.j_entry[e];
                    const uint2 ab = d.jq_ab[g.q0 + en.x];
                    const JointRec r = {d.jq_anchor[g.q0 + en.x], d.jq_mass[g.q0 + en.x], d.jq_len[g.q0 + en.x].x,
                                        ab.x, ab.y};
                    d.jrot[en.y] = solve(r, [&](uint32_t i) { return d.b.pos[d.jg_body[g.b0 + i]]; },
                                         [&](uint32_t i, float2 p) { d.b.pos[d.jg_body[g.b0 + i]] = p; });
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // memory: wait for the writes
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
    if (flags) atomicOr(&d.accum->error_flags, flags);
    __syncthreads();
    if (staged)
        for (uint32_t i = tid; i < nbod; i += NT) d.b.pos[s_gid[i]] = s_pos[i];
    for (uint32_t e = tid; e < n; e += NT) {
        const uint2 en = staged ? s_entry[e] : d.j_entry[e0 + e];
        const float2 axis = staged ? s_axis[e] : d.jrot[en.y];
        const float target = staged ? s_len[en.x].y : d.jq_len[g.q0 + en.x].y;
        float2 step = make_float2(0.0f, 0.0f);  // coincident anchors: the reference skips the solve
        if (!(vlen(axis.x, axis.y) < 1e-6f)) step = make_float2(joint_rotation_corr(axis.x, axis.y, target) * h, 1.0f);
        d.jrot[en.y] = step;
    }
}

__global__ __launch_bounds__(kJointThreads) void k_joints(DeviceWorld d, float h) {
    __shared__ JointsLds lds;
    joint_group<kJointThreads>(d, h, blockIdx.x, lds);
}

// Verlet + collider transforms + constraints (physics.rs:323-395), and the
// bounding box of the colliders for the next substep's grid.  kBodyLanes lanes
// a body: each works the body out (they load the same lines) and transforms
// every kBodyLanes-th of its colliders, the first of which it loads beside the
// body, so that 65,536 bodies are four waves a SIMD and not one: 18.9 us with
// 294,249 colliders against 24.9 (6.0 against 10.4 at 250 bodies).
constexpr uint32_t kBodyLanes = 4;

struct Box {
    uint32_t b0 = 0xFFFFFFFFu, b1 = 0xFFFFFFFFu, b2 = 0u, b3 = 0u;  // f2ord bounding box
};
// (whole waves: thread t of the pass)
__device__ __forceinline__ void integrate_at(const DeviceWorld& d, const SubstepArgs& a, uint32_t t, Box& box) {
    const uint32_t b = t / kBodyLanes, r = t % kBodyLanes;
    uint32_t flags = 0;
    if (b < d.nb) {
        const uint32_t fl = d.b.bflags[b];
        const uint32_t c0 = d.bc_start[b], c1 = d.bc_start[b + 1];
        BodyState s;
        s.p = d.b.pos[b];
        s.po = d.b.pos_old[b];
        s.rot = d.b.rot[b];
        s.omega = d.b.omega[b];
        uint32_t e0 = 0, n = 0;
        if (a.joint_rot) {
            e0 = d.bj_start[b];
            n = d.bj_start[b + 1] - e0;
        }
        uint32_t c = 0;
        float2 off = make_float2(0.0f, 0.0f);
        if (c0 + r < c1) {
            c = d.bc_list[c0 + r];
            off = d.c.off[c];
        }
        const float rot_in = s.rot;
        {
            // this body's joint rotation steps (physics.rs:468-469), in the order of the sweep:
            // iterations, then joints in arena order; a few load at a time
            const uint32_t total = n * a.joint_iters;
            uint32_t i = 0, it = 0;  // position m is entry i of iteration it
            for (uint32_t m = 0; m < total; m += 4) {
                uint32_t ent[4];
                float2 step[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) {
                    ent[u] = d.bj_list[e0 + i];
                    step[u] = d.jrot[(size_t)it * a.joint_count + (ent[u] >> 1)];
                    if (m + u + 1 < total && ++i == n) {
                        i = 0;
                        ++it;
                    }
                }
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) {
                    if (m + u >= total || step[u].y == 0.0f) continue;
                    s.rot = (ent[u] & 1u) ? s.rot - step[u].x : s.rot + step[u].x;
                    if (!finitef(s.rot)) flags |= ERR_JOINT_ROT;
                }
            }
        }
        const float om0 = s.omega;
        if (fl & BF_STATIC) {  // :327-332
            s.po = s.p;
            s.vel = make_float2(0.0f, 0.0f);
        } else {
            float2 acc;
            if (a.has_springs) {
                acc = d.b.acc[b];
            } else {
                acc = a.fresh ? d.b.acc[b] : make_float2(0.0f, 0.0f);
                float gm = d.b.gmod[b];
                acc.x = acc.x + a.gx * gm;
                acc.y = acc.y + a.gy * gm;
            }
            const bool vr = fl & BF_HAS_VREQ;
            float2 vreq = vr ? d.b.vreq[b] : make_float2(0.0f, 0.0f);
            float tq = a.fresh ? d.b.torque[b] : 0.0f;
            float toi = (a.fresh || !(fl & BF_INERTIA_POS)) ? tq / d.b.inertia[b] : 0.0f;
            float ratio = a.ratio_rest;
            if ((int32_t)b == a.first_dyn) ratio = a.h / d.accum->old_dt;
            verlet_dynamic(s, acc, toi, vr, vreq, a.h, ratio);
        }
        // collider transforms from the pre-constraint position (:360-366)
        if (c0 + r < c1) {
            float sn, cs;
            rot_sincos(s.rot, &sn, &cs);
            for (uint32_t k = c0 + r;;) {
                const float2 x = body_xform(sn, cs, s.p, off);
                d.c.abs[c] = x;
                if (finitef(x.x) && finitef(x.y)) {
                    box.b0 = min(box.b0, f2ord(x.x));
                    box.b1 = min(box.b1, f2ord(x.y));
                    box.b2 = max(box.b2, f2ord(x.x));
                    box.b3 = max(box.b3, f2ord(x.y));
                }
                k += kBodyLanes;
                if (k >= c1) break;
                c = d.bc_list[k];
                off = d.c.off[c];
            }
        }
        apply_constraints(s.p, d.con_pos, d.con_r, d.nk);
        // a wave holds whole bodies and runs in step: every lane has read its body by now
        __builtin_amdgcn_wave_barrier();
        if (r == 0) {
            d.b.pos[b] = s.p;
            d.b.pos_old[b] = s.po;
            d.b.vel[b] = s.vel;
            if (__float_as_uint(s.rot) != __float_as_uint(rot_in)) d.b.rot[b] = s.rot;
            if (__float_as_uint(s.omega) != __float_as_uint(om0)) d.b.omega[b] = s.omega;
            if (!(fl & BF_STATIC)) {
                if (fl & BF_HAS_VREQ) d.b.bflags[b] = fl & ~BF_HAS_VREQ;
                if (a.fresh) d.b.torque[b] = 0.0f;
                if ((int32_t)b == a.first_dyn) d.accum->old_dt = a.h;
            }
        }
    }
    static_assert(BG_WAVE % kBodyLanes == 0, "a body's lanes in one wave");
    if (flags) atomicOr(&d.accum->error_flags, flags);
}
// The block's box into the substep's record.
template <uint32_t NT>
__device__ __forceinline__ void box_flush(const DeviceWorld& d, uint32_t parity, const Box& box,
                                          uint32_t (&s_box)[4][NT / BG_WAVE]) {
    const uint32_t b0 = wave_prefix(box.b0, 0xFFFFFFFFu, MinU32());
    const uint32_t b1 = wave_prefix(box.b1, 0xFFFFFFFFu, MinU32());
    const uint32_t b2 = wave_prefix(box.b2, 0u, MaxU32());
    const uint32_t b3 = wave_prefix(box.b3, 0u, MaxU32());
    const uint32_t wv = threadIdx.x / BG_WAVE;
    if ((threadIdx.x & (BG_WAVE - 1)) == BG_WAVE - 1) {
        s_box[0][wv] = b0;
        s_box[1][wv] = b1;
        s_box[2][wv] = b2;
        s_box[3][wv] = b3;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        const uint32_t* v = s_box[threadIdx.x];
        uint32_t* to = &d.accum->bbox[parity][threadIdx.x];
        uint32_t m = v[0];
#pragma unroll
        for (uint32_t i = 1; i < NT / BG_WAVE; ++i) m = threadIdx.x < 2 ? min(m, v[i]) : max(m, v[i]);
        if (threadIdx.x < 2)
            atomic_min_if_less(to, m);
        else
            atomic_max_if_greater(to, m);
    }
}

__global__ __launch_bounds__(kThreads) void k_integrate(DeviceWorld d, SubstepArgs a) {
    __shared__ uint32_t s_box[4][kThreads / BG_WAVE];
    Box box;
    integrate_at(d, a, blockIdx.x * blockDim.x + threadIdx.x, box);
    box_flush<kThreads>(d, a.parity, box, s_box);
}

// ---- small worlds ------------------------------------------------------------
//
// A world of at most kSmallColliders colliders and kSmallGeneral bodies takes its substep in four
// launches instead of ten: one workgroup sorts and works out the contacts, one solves the
// joints and integrates (the fallback and the ordered pass in between, which have nothing to do
// in most substeps).  A pass of such a world is a launch's few microseconds whatever it does, and
// a barrier a tenth of one; but one workgroup has one CU's latency to hide its loads in, and each
// further round over the colliders (1,024 a round) or the bodies (256, at four lanes each) costs part
// of what the launches did.  A step in one workgroup against ten launches, us:
//   48 bodies 273 / 330, 120 301 / 360, 200 329 / 371;
//   256 bodies of  256 colliders 292 / 344,   512 303 / 352,   817 322 / 364, 1,024 354 / 450,
//              1,152 386 / 464, 1,216 408 / 471, 1,280 445 / 492, 1,408 575 / 569, 1,536 734 / 658;
//   128 bodies of 1,000 746 / 777, 1,100 906 / 896, 1,152 1,027 / 995, 1,280 1,305 / 1,238;
//   past 256 bodies: 262 of 1,152 406 / 382, 300 442 / 389, 320 of 320 359 / 361, 512 of 512 411 / 366.
// So the bodies stop at one round.  The colliders' second round still pays up to some 1,400 where a body
// has few of them, and from 1,100 on no longer at nine a body: the limit lies between the two.
constexpr uint32_t kSmallThreads = 1024;

template <bool GROUPS, bool SENSORS>
__global__ __launch_bounds__(kSmallThreads) void k_small_contacts(KeysArgs k, CellScatter sc, DeviceWorld d,
                                                                  SubstepArgs a) {
    __shared__ ListsLds lds[kSmallThreads / BG_WAVE];
    __shared__ uint32_t red[kSmallThreads / BG_WAVE];
    const uint32_t t = threadIdx.x;
    for (uint32_t i = t; i < d.nc + (a.has_springs ? d.nb : 0u); i += kSmallThreads) {
        if (i < d.nc)
            rebuild_key_at<false>(i, k);
        else
            forces_at(i - d.nc, d, a);
    }
    __syncthreads();
    {  // exclusive scan of the cells' counts, which are cleared: up to four times four a thread
        const uint32_t n = d.grid->ncells, n4 = (n + 3u) / 4u, per = (n4 + kSmallThreads - 1u) / kSmallThreads;
        uint4* cnt = reinterpret_cast<uint4*>(k.cnt);
        uint4* start = reinterpret_cast<uint4*>(d.cell_start);
        uint4 v[4];
        uint32_t sum = 0;
#pragma unroll
        for (uint32_t g = 0; g < 4; ++g) {
            const uint32_t i = t * per + g;
            v[g] = g < per && i < n4 ? cnt[i] : make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (uint32_t g = 0; g < 4; ++g) sum += v[g].x + v[g].y + v[g].z + v[g].w;
        const uint32_t incl = wave_prefix(sum, 0u, AddU32()), lane = t & (BG_WAVE - 1);
        if (lane == BG_WAVE - 1) red[t / BG_WAVE] = incl;
        __syncthreads();
        const uint32_t tot = wave_prefix(lane < kSmallThreads / BG_WAVE ? red[lane] : 0u, 0u, AddU32());
        const int w = __builtin_amdgcn_readfirstlane((int)(t / BG_WAVE));
        uint32_t run = (w > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)tot, w - 1) : 0u) + incl - sum;
#pragma unroll
        for (uint32_t g = 0; g < 4; ++g) {
            const uint32_t i = t * per + g;
            if (g >= per || i >= n4) continue;
            const uint4 c = v[g];
            start[i] = make_uint4(run, run + c.x, run + c.x + c.y, run + c.x + c.y + c.z);
            run += c.x + c.y + c.z + c.w;
            cnt[i] = make_uint4(0u, 0u, 0u, 0u);
        }
        __syncthreads();
        if (t == 0) d.cell_start[n] = d.nc;  // (the table has a word to spare)
        static_assert(kSmallColliders * 4u <= 16u * kSmallThreads, "cells of the largest: next power of two of four a collider");
    }
    __syncthreads();
    for (uint32_t i = t; i < d.nc; i += kSmallThreads) scatter_at(i, sc);
    __syncthreads();
    for (uint32_t i = t; i < (d.nc + BG_WAVE - 1u) / BG_WAVE * BG_WAVE; i += kSmallThreads)
        contact_lists<GROUPS, SENSORS>(d, a, lds[t / BG_WAVE], i, i / BG_WAVE);
    __syncthreads();
    for (uint32_t i = t; i < (d.nb * kMergeLanes + BG_WAVE - 1u) / BG_WAVE * BG_WAVE; i += kSmallThreads)
        contact_merge(d, i);
}

__global__ __launch_bounds__(kSmallThreads) void k_small_integrate(DeviceWorld d, SubstepArgs a) {
    __shared__ JointsLds lds;
    __shared__ uint32_t s_box[4][kSmallThreads / BG_WAVE];
    if (a.joint_rot)
        for (uint32_t g = 0; g < d.n_jgroups; ++g) {
            joint_group<kSmallThreads>(d, a.h, g, lds);
            __syncthreads();
        }
    Box box;
    for (uint32_t i = threadIdx.x; i < (d.nb * kBodyLanes + BG_WAVE - 1u) / BG_WAVE * BG_WAVE; i += kSmallThreads)
        integrate_at(d, a, i, box);
    box_flush<kSmallThreads>(d, a.parity, box, s_box);
}

}  // namespace

// ============================================================ launchers

// Counting sort by cell: cell_start = exclusive scan of the counts of the
// fitted grid's cells (cell_start[ncells] = nc), then the scatter.
hipError_t launch_rebuild_sort_and_cells(DeviceWorld& d) {
    // the grid the key pass fitted holds ncells <= cells_cap cells: the scan covers those
    // (the count is read on the device), not the whole table
    const uint32_t* last =
        reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(d.grid) + offsetof(GridParams, ncells));
    hipError_t e = exclusive_scan_u32(d.cell_count, d.cell_start, d.cells_cap + 1, d.sort, d.stream, last);
    if (e != hipSuccess) return e;
    const uint32_t n = d.nc > 0 ? d.nc : 1u;
    k_cell_scatter<<<div_up(n, kThreads), kThreads, 0, d.stream>>>(cell_scatter_of(d), d.cell_count, d.cells_cap + 1,
                                                                   d.grid, d.accum);
    return hipGetLastError();
}

hipError_t launch_general_substep(DeviceWorld& d, const SubstepArgs& a, bool groups, bool sensors,
                                  const KeysArgs* rebuild) {
    if (d.nb == 0) return hipSuccess;
    const uint32_t blocks = div_up(d.nb, kThreads);
    const bool small = rebuild && a.collisions && d.clist && d.nc > 0 && d.nc <= kSmallColliders && d.nb <= kSmallGeneral;
    SubstepArgs ai = a;
    ai.joint_rot = 0u;
    if (d.n_jgroups > 0 && d.j_iters > 0) {
        ai.joint_rot = 1u;
        ai.joint_iters = d.j_iters;
        ai.joint_count = d.nj;
    }
    if (small) {
        const CellScatter sc = cell_scatter_of(d);
        const uint32_t fb = std::min(div_up(d.nb, kContactThreads), 256u);
#define BG_SMALL(G, S)                                                                  \
    do {                                                                                \
        k_small_contacts<G, S><<<1, kSmallThreads, 0, d.stream>>>(*rebuild, sc, d, a);  \
        k_contacts<G, S><<<fb, kContactThreads, 0, d.stream>>>(d, a, d.cfb_list);       \
    } while (0)
        if (groups && sensors)
            BG_SMALL(true, true);
        else if (groups)
            BG_SMALL(true, false);
        else if (sensors)
            BG_SMALL(false, true);
        else
            BG_SMALL(false, false);
#undef BG_SMALL
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        e = launch_contacts_ordered(d, a, groups, sensors);
        if (e != hipSuccess) return e;
        k_small_integrate<<<1, kSmallThreads, 0, d.stream>>>(d, ai);
        return hipGetLastError();
    }
    // the rebuild's keys and the substep's forces in one launch, then the rest of the rebuild
    const uint32_t key_blocks = rebuild ? div_up(rebuild->nc > 0 ? rebuild->nc : 1u, kThreads) : 0u;
    const uint32_t force_blocks = a.has_springs ? blocks : 0u;
    if (key_blocks + force_blocks > 0)
        k_keys_forces<<<key_blocks + force_blocks, kThreads, 0, d.stream>>>(rebuild ? *rebuild : KeysArgs{},
                                                                            key_blocks, d, a);
    if (rebuild) {
        hipError_t e = launch_rebuild_sort_and_cells(d);
        if (e != hipSuccess) return e;
    }
    if (a.collisions && d.nc > 0) {
        // One-wave blocks: a body's work varies with its collider count, so small blocks
        // keep the slow waves from holding whole workgroups.  With the collider lists
        // allocated: one thread per collider, a per-body merge, and the full per-body
        // walk only for the bodies the merge could not take.
        const uint32_t cb = div_up(d.nb, kContactThreads);
#define BG_CONTACTS(G, S)                                                                                     \
    do {                                                                                                      \
        if (d.clist) {                                                                                        \
            k_contact_lists<G, S><<<div_up(d.nc, kContactThreads), kContactThreads, 0, d.stream>>>(d, a);     \
            k_contact_merge<<<div_up(d.nb, kThreads / kMergeLanes), kThreads, 0, d.stream>>>(d);              \
            k_contacts<G, S><<<std::min(cb, 256u), kContactThreads, 0, d.stream>>>(d, a, d.cfb_list);         \
        } else {                                                                                              \
            k_contacts<G, S><<<cb, kContactThreads, 0, d.stream>>>(d, a, nullptr);                            \
        }                                                                                                     \
    } while (0)
        if (groups && sensors)
            BG_CONTACTS(true, true);
        else if (groups)
            BG_CONTACTS(true, false);
        else if (sensors)
            BG_CONTACTS(false, true);
        else
            BG_CONTACTS(false, false);
#undef BG_CONTACTS
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        e = launch_contacts_ordered(d, a, groups, sensors);
        if (e != hipSuccess) return e;
    }
    if (ai.joint_rot) k_joints<<<d.n_jgroups, kJointThreads, 0, d.stream>>>(d, a.h);
    k_integrate<<<div_up(d.nb, kThreads / kBodyLanes), kThreads, 0, d.stream>>>(d, ai);
    return hipGetLastError();
}

}  // namespace bg
