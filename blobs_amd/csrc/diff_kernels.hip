// diff_kernels.hip -- forward and adjoint of rollouts of single-sphere worlds
// with springs, one workgroup per world for a whole segment of steps: a body a
// thread and as few threads as hold the largest world (256, 512, 1,024; two
// bodies a thread past that).  Positions, velocities, partner lists, the spring
// forces, the joint records and the adjoint vectors live in LDS.
//
// Forward substep (physics.rs:401-421, same f32 operation order as the
// general path): gravity and springs per body in ascending spring index
// (springs.rs:25-47), contacts against the substep's snapshot summed in
// ascending partner index (physics.rs:241-317), Verlet (physics.rs:323-358),
// collider transform = position (zero offsets).
//
// A world has one workgroup, so a launch takes what its slowest world takes
// and a substep is bound by VALU issue and by its chain of phases (a barrier
// between them).  Hence contacts worked out from a queue by all threads;
// springs evaluated once each by a thread of their own (at most
// kDiffLdsSprings; a body then sums its springs' terms from LDS in ascending
// index); joints swept level by level on records staged in LDS
// (joint_schedule.hpp); and the next tape slot loaded while the reverse works
// on the current one.  Recompute and reverse are kernels of their own: in one,
// their state spilled 55 VGPRs.
//
// Partner lists.  Most bodies of such worlds move a thousandth of a diameter a
// substep and a few a twentieth, so a list of the bodies within two skins of
// reach serves for tens of substeps.  A body is in reach of another only if
// the two paths since the build, the world's mean motion taken out, add up to
// the rest, so a body whose path exceeds the skin leaves the lists and is tested
// by everyone (its own pairs come from those tests), until the tests cost as
// much as a build.  A world too dense for lists is filed by cell every substep.
//
// Measured (forward + backward, against bounding box, grid, springs and contacts
// worked out serially or per body each substep; in brackets with a grid and
// 1,024 threads for every world in every substep): 256 worlds of 2,048 bodies and
// 1,024 springs over 50 steps 33.2 -> 14.5 ms (15.4); 96 worlds of 700, 60 steps
// forward 7.24 -> 2.68 ms (3.13); 12 worlds of 301 with 40 joints, 6 steps 3.80 ->
// 1.53 ms (1.61); 512 worlds of 300, 20 steps 1.10 ms (1.98).
#include "diff.hpp"

#include <algorithm>

#include "lds_grid.hpp"

namespace bg {

namespace {

// A world's workgroup: NT threads, PER bodies a thread.
template <uint32_t NT, uint32_t PER>
struct Rollout {
static constexpr uint32_t kDiffThreads = NT, kDiffMaxBodies = NT * PER;
static constexpr uint32_t kDiffCells = PER == 1 ? 2 * NT : 3 * NT;
static constexpr uint32_t kPairs = PER == 1 ? NT + NT / 4 : 1200;  // queued contact pairs of a substep
static constexpr int kWaves = NT / BG_WAVE;
static constexpr uint32_t kScanItems = (kDiffCells + 1 + kDiffThreads - 1) / kDiffThreads;
// Springs of a world whose terms are kept in LDS (32 KB of it); a world with more evaluates
// them per body.
static constexpr uint32_t kDiffLdsSprings = 2048;
// A world whose joint records and schedule are staged in LDS has at most so many joints,
// solves a substep and levels of them.
static constexpr uint32_t kDiffLdsJoints = 256, kDiffLdsSolves = NT, kDiffLdsLevels = 512;
// Partner lists: entries of a body, bodies outside the lists and queued pairs of each, builds with
// the skin halved while too many lists overflow, and the substeps a world that overflows them all
// goes without.  The skin in diameters of the largest body: with 0.1 the four cases above take
// 15.6, 3.03, 1.50 and 1.17 ms, with 0.3 16.3, 2.79, 1.54 and 1.11, with 0.2 14.8, 2.66, 1.53 and 1.10.
static constexpr uint32_t kListCap = 8, kOutMax = 16, kOutPairs = 8, kListTries = 3, kGridHold = 64;
static constexpr float kSkin = 0.2f;
static constexpr uint32_t kTested = 24;           // a build costs about what so many tests of a body outside the lists do
static constexpr uint32_t kOut = 15;              // Own::nl of a body outside the lists
static_assert(kDiffLdsSolves <= kDiffThreads, "a thread stages one axis");
static constexpr uint32_t kKept = 16;             // partners of a body that queue_rounds remembers
static constexpr uint32_t kInc = 4;               // springs of a body kept as packed registers

struct JointRec {
    float4 anchor;  // a (x, y), b (z, w)
    float4 mass;    // 1/m_a + 1/m_b, ratio, 1 - ratio, distance
    uint32_t ab;    // local a | a is static << 15 | local b << 16 | b is static << 31
};
struct JointStage {
    float4 anchor[kDiffLdsJoints], mass[kDiffLdsJoints];
    uint32_t ab[kDiffLdsJoints];
    uint16_t entry[kDiffLdsSolves], level[kDiffLdsLevels + 1];
};

// Bodies outside the lists, by substep parity where a phase clears what another reads.
struct Outliers {
    uint32_t n;           // (may exceed kOutMax: then the lists are built anew)
    uint32_t pairs[2];    // queued pairs
    uint32_t round, more; // and of a round of queue_rounds; somebody has contacts left
    uint16_t id[kOutMax];
    uint32_t count[2][kOutMax];  // pairs of an outlier, in the queue's entries from kPairs + u * kOutPairs
};
// The lists' state, the same in every thread.
struct Walk {
    float skin;
    float2 drift;  // the world's common motion a substep
    uint32_t grid; // substeps left without lists
    uint32_t tested;  // bodies outside the lists, summed over the substeps since the build
    bool build;
};

struct Ctx {
    float2* xy;        // positions (the snapshot)
    float2* vel;       // calculated_velocity
    float* mass;
    float* rad;        // radii
    float4* rec;       // bodies in cell order (the memory of `force` or of `lists`); the reverse's
                       // snapshot (x, y, radius, mass) by index
    uint16_t (*lists)[kDiffMaxBodies][4];  // [kListCap / 4]: partners by body; forward only
    float2* res;       // [kPairs] corrections of the queue; forward only
    uint32_t* entries; // [kPairs] its pairs
    Outliers* out;
    float* gmod;       // gravity_mod; forward only
    uint32_t* cnt;     // [kDiffCells + 1] cell counts, then cell starts; forward only
    float2 *spring_k, *spring_v;  // spring adjoints; reverse only
    float4* force;     // per spring: (Fx / m_a, Fy / m_a, -Fx / m_b, -Fy / m_b); forward only
    uint32_t* red;     // [kFitWords][kWaves]
    double* dred;      // [2][kWaves]
    LdsGrid* grid;
    JointStage* joints;  // of a staged world
    float2* axes;        // its solves' axes; reverse only
    float2* lam_pp;    // adjoint only (the memory of `force`)
    float2* lam_am;
};

// A thread's two bodies.  The phases loop over them at run time and pick the state by
// selects: unrolled, two bodies' contact passes in flight spill 50 to 140 VGPRs.
struct Own {
    float2 p[PER], q[PER];
    float travel[PER];            // path since the lists were built, the common motion taken out
    uint32_t nl;                // list lengths, four bits each (kOut: outside the lists)
    uint32_t fl[PER];             // body flags | springs of the body << 8 (at most kIncMany: more are counted anew)
    uint32_t inc0[PER], inc1[PER];  // first kInc springs, two a word: local spring << 1 | (1: the body is its b)
    // the spring this thread evaluates first
    uint32_t s_ab;
    float s_rest, s_k, s_c;
};
static constexpr uint32_t kIncMany = 0xFFFFFFu;
static_assert(PER == 1 || PER == 2, "the picks");
static __device__ __forceinline__ uint32_t per_thread(const DiffWorld& W) { return PER == 1 || W.nb <= NT ? 1u : 2u; }

// The thread's index, opaque to the compiler: the phases of a substep recompute what they
// derive from it, where hoisted out of the substep loop those addresses spill.
static __device__ __forceinline__ uint32_t thread_index() {
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

static __device__ __forceinline__ bool lds_springs(const DiffWorld& W) { return W.ns <= kDiffLdsSprings; }

static __device__ __forceinline__ bool joints_staged(const DiffWorld& W) {
    return W.njq <= kDiffLdsJoints && W.nje <= kDiffLdsSolves && W.njl <= kDiffLdsLevels;
}

// Joint q of the world: from LDS in a staged world, else from global memory.  (Templates:
// where the two meet in one load it becomes a flat one.)
template <bool STAGED>
static __device__ __forceinline__ JointRec joint_rec(const Ctx& c, const DiffArgs& a, const DiffWorld& W, uint32_t q) {
    JointRec r;
    if constexpr (STAGED) {
        r.anchor = c.joints->anchor[q];
        r.mass = c.joints->mass[q];
        r.ab = c.joints->ab[q];
    } else {
        r.anchor = a.j_anchor[W.jq0 + q];
        r.mass = a.j_mass[W.jq0 + q];
        r.mass.w = a.j_dist[W.jq0 + q];
        r.ab = a.j_ab[W.jq0 + q];
    }
    return r;
}
static_assert(kDiffMaxBodies <= 0x7FFF, "15-bit body indices in JointRec::ab");

// Runs the world's joint solves level by level, a wave a group: solve(e, record) for solve e
// of the world.  REVERSE: from the last level to the first.  The next level's records load
// while the current one works.
template <bool STAGED, bool REVERSE, class Solve>
static __device__ __forceinline__ void joint_levels(const Ctx& c, const DiffArgs& a, const DiffWorld& W, Solve&& solve) {
    const uint32_t lane = threadIdx.x & (BG_WAVE - 1);
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / BG_WAVE));
    for (uint32_t grp = W.jg0 + wave; grp < W.jg0 + W.njg; grp += kWaves) {
        const uint32_t l0 = a.jg_level[grp] - W.jl0, n = a.jg_level[grp + 1] - W.jl0 - l0;
        uint32_t e, q;
        JointRec r;
        bool have;
        auto load = [&](uint32_t k) {
            const uint32_t l = l0 + (REVERSE ? n - 1u - k : k);
            uint32_t end;
            if constexpr (STAGED) {
                e = c.joints->level[l] + lane;
                end = c.joints->level[l + 1];
            } else {
                e = a.jl_start[W.jl0 + l] - W.je0 + lane;
                end = a.jl_start[W.jl0 + l + 1] - W.je0;
            }
            have = e < end;
            if (!have) return;
            if constexpr (STAGED)
                q = c.joints->entry[e];
            else
                q = a.j_entry[W.je0 + e];
            r = joint_rec<STAGED>(c, a, W, q);
        };
        if (n > 0) load(0);
        for (uint32_t k = 0; k < n; ++k) {
            const uint32_t e_now = e;
            const JointRec r_now = r;
            const bool have_now = have;
            if (k + 1 < n) load(k + 1);
            if (have_now) solve(e_now, r_now);
            // the next level's lanes read what this one's wrote: one wave's LDS accesses keep
            // their order, the compiler has to as well
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

static __device__ __forceinline__ void load_own(Ctx& c, Own& o, const DiffArgs& a, const DiffWorld& W, const float2* p,
                                         const float2* q, const float2* v) {
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        const uint32_t li = threadIdx.x + j * kDiffThreads;
        const bool live = li < W.nb;
        const uint32_t g = W.b0 + (live ? li : 0u);
        o.p[j] = live ? p[g] : make_float2(0.0f, 0.0f);
        o.q[j] = live ? q[g] : make_float2(0.0f, 0.0f);
        o.travel[j] = 0.0f;
        o.fl[j] = a.flags[g] & 0xFFu;
        o.inc0[j] = o.inc1[j] = 0;
        if (!live) continue;
        c.xy[li] = o.p[j];
        c.vel[li] = v[g];
        c.mass[li] = a.mass[g];
        c.rad[li] = a.radius[g];
        if (c.gmod) c.gmod[li] = a.gmod[g];
        const uint32_t e0 = a.inc_start[g], n_inc = a.inc_start[g + 1] - e0;
        o.fl[j] |= min(n_inc, kIncMany) << 8;
        if (lds_springs(W)) {
#pragma unroll
            for (uint32_t t = 0; t < kInc; ++t)
                if (t < n_inc) {
                    const uint32_t s = a.inc_list[e0 + t];
                    const uint32_t e = ((s - W.s0) << 1) | ((uint32_t)a.sp_a[s] == g ? 0u : 1u);
                    (t < 2 ? o.inc0[j] : o.inc1[j]) |= e << (16u * (t & 1u));
                }
        }
    }
    o.nl = 0;
    o.s_ab = 0;
    o.s_rest = o.s_k = o.s_c = 0.0f;
    if (threadIdx.x < W.ns) {
        const uint32_t s = W.s0 + threadIdx.x;
        o.s_ab = ((uint32_t)a.sp_a[s] - W.b0) | (((uint32_t)a.sp_b[s] - W.b0) << 16);
        o.s_rest = a.sp_rest[s];
        o.s_k = a.sp_k[s];
        o.s_c = a.sp_c[s];
    }
    if (W.njg > 0 && joints_staged(W)) {
        for (uint32_t k = threadIdx.x; k < W.njq; k += kDiffThreads) {
            const JointRec r = joint_rec<false>(c, a, W, k);
            c.joints->anchor[k] = r.anchor;
            c.joints->mass[k] = r.mass;
            c.joints->ab[k] = r.ab;
        }
        for (uint32_t k = threadIdx.x; k < W.nje; k += kDiffThreads)
            c.joints->entry[k] = (uint16_t)a.j_entry[W.je0 + k];
        for (uint32_t k = threadIdx.x; k <= W.njl; k += kDiffThreads)
            c.joints->level[k] = (uint16_t)(a.jl_start[W.jl0 + k] - W.je0);
    }
}

// f(incidence) over body j's springs in ascending index; incidence as in Own::inc0.
template <class F>
static __device__ __forceinline__ void for_springs(const Own& o, uint32_t j, const DiffArgs& a, const DiffWorld& W, F&& f) {
    const uint32_t n = pick(o.fl, j) >> 8, w0 = pick(o.inc0, j), w1 = pick(o.inc1, j);
    if (n > 0) f(w0 & 0xFFFFu);
    if (n > 1) f(w0 >> 16);
    if (n > 2) f(w1 & 0xFFFFu);
    if (n > 3) f(w1 >> 16);
    static_assert(kInc == 4, "the four above");
    if (n > kInc) {
        const uint32_t g = W.b0 + threadIdx.x + j * kDiffThreads, e0 = a.inc_start[g], e1 = a.inc_start[g + 1];
        for (uint32_t t = kInc; t < e1 - e0; ++t) {
            const uint32_t s = a.inc_list[e0 + t];
            f(((s - W.s0) << 1) | ((uint32_t)a.sp_a[s] == g ? 0u : 1u));
        }
    }
}

// f(local spring, local a, local b, rest, k, c) over the springs this thread evaluates.
template <class F>
static __device__ __forceinline__ void own_springs(const Own& o, const DiffArgs& a, const DiffWorld& W, F&& f) {
    uint32_t ab = o.s_ab;
    float rest = o.s_rest, k = o.s_k, cc = o.s_c;
    for (uint32_t t = threadIdx.x; t < W.ns;) {
        f(t, ab & 0xFFFFu, ab >> 16, rest, k, cc);
        t += kDiffThreads;
        if (t < W.ns) {
            const uint32_t s = W.s0 + t;
            ab = ((uint32_t)a.sp_a[s] - W.b0) | (((uint32_t)a.sp_b[s] - W.b0) << 16);
            rest = a.sp_rest[s];
            k = a.sp_k[s];
            cc = a.sp_c[s];
        }
    }
}

// Force of one spring on its body a (springs.rs:25-47); -F acts on b.
static __device__ __forceinline__ float2 spring_force(float2 pa, float2 pb, float2 va, float2 vb, float rest, float k, float c) {
    const float dx = pb.x - pa.x, dy = pb.y - pa.y;
    const float dist = vlen(dx, dy);
    const float ux = dx / dist, uy = dy / dist;
    const float rvx = va.x - vb.x, rvy = va.y - vb.y;
    const float dot = rvx * ux + rvy * uy;
    const float cd = c * dot;
    const float dfx = cd * ux, dfy = cd * uy;
    const float mag = k * (dist - rest);
    return make_float2(ux * (mag - dfx), uy * (mag - dfy));
}

// Position sweep of the world's joints (physics.rs:426-460) on the LDS positions P; with REC
// every solve's anchor axis is recorded.
template <bool REC, bool STAGED>
static __device__ __forceinline__ void joint_sweep(Ctx& c, float2* P, const DiffArgs& a, const DiffWorld& W, uint32_t slot) {
    uint32_t flags = 0;
    joint_levels<STAGED, false>(c, a, W, [&](uint32_t e, const JointRec& r) {
        const uint32_t la = r.ab & 0x7FFFu, lb = (r.ab >> 16) & 0x7FFFu;
        float2 pa = P[la], pb = P[lb];
        float dx, dy;
        const bool moved =
            joint_positions(pa, pb, make_float2(r.anchor.x, r.anchor.y), make_float2(r.anchor.z, r.anchor.w), r.mass.w,
                            make_float4(r.mass.x, r.mass.y, r.mass.z, 1.0f), (r.ab & (1u << 15)) != 0u,
                            (r.ab & (1u << 31)) != 0u, dx, dy, flags);
        if (REC) a.tape_axis[(size_t)slot * a.n_solves + W.je0 + e] = make_float2(dx, dy);
        if (!moved) return;
        P[la] = pa;
        P[lb] = pb;
    });
}

// Adjoint of joint_sweep on the LDS position adjoints L, from the axes the
// forward sweep recorded: last solve first.
template <bool STAGED>
static __device__ __forceinline__ void joint_sweep_reverse(Ctx& c, float2* L, const DiffArgs& a, const DiffWorld& W,
                                                    uint32_t slot) {
    joint_levels<STAGED, true>(c, a, W, [&](uint32_t e, const JointRec& r) {
        float2 d;
        if constexpr (STAGED)
            d = c.axes[e];
        else
            d = a.tape_axis[(size_t)slot * a.n_solves + W.je0 + e];
        const float dist = vlen(d.x, d.y);
        if (dist < 1e-6f) return;  // the reference skips the joint
        const uint32_t la = r.ab & 0x7FFFu, lb = (r.ab >> 16) & 0x7FFFu;
        const bool sa = (r.ab & (1u << 15)) != 0u, sb = (r.ab & (1u << 31)) != 0u;
        // weights (physics.rs:450-460): a static -> b moves by ims corr; b static -> a does;
        // otherwise a by ratio corr and b by (1 - ratio) corr
        const float wa = sa ? 0.0f : (sb ? r.mass.x : r.mass.y);
        const float wb = sa ? r.mass.x : (sb ? 0.0f : r.mass.z);
        const float2 la2 = L[la], lb2 = L[lb];
        const float lcx = wa * la2.x - wb * lb2.x, lcy = wa * la2.y - wb * lb2.y;
        const float nx = d.x / dist, ny = d.y / dist;
        const float nm = nx * lcx + ny * lcy;
        const float f = r.mass.w / dist;
        const float ldx = lcx - f * (lcx - nx * nm), ldy = lcy - f * (lcy - ny * nm);
        L[la] = make_float2(la2.x - ldx, la2.y - ldy);
        L[lb] = make_float2(lb2.x + ldx, lb2.y + ldy);
    });
}

// update_objects of body j (physics.rs:326-358) from its position after the contact and joint
// stages; the snapshot is the new position.
static __device__ __forceinline__ void verlet(Ctx& c, Own& o, const Walk& w, const DiffArgs& a, const DiffWorld& W,
                                       uint32_t gsub, uint32_t j, float2 pn, float2 acc) {
    const uint32_t tid = thread_index();
    const float h = a.h;
    const uint32_t li = tid + j * kDiffThreads, fl = pick(o.fl, j);
    BodyState st;
    st.p = pn;
    st.po = pick(o.q, j);
    st.rot = 0.0f;
    st.omega = 0.0f;
    if (fl & BF_STATIC) {
        st.po = pn;
        st.vel = make_float2(0.0f, 0.0f);
    } else {
        const bool vr = gsub == 0 && (fl & BF_HAS_VREQ);
        const float2 vq = vr ? a.vreq[W.b0 + li] : make_float2(0.0f, 0.0f);
        const float ratio = ((int32_t)li == W.first_dyn && gsub == 0) ? h / W.old_dt0 : h / h;
        verlet_dynamic(st, acc, 0.0f, vr, vq, h, ratio);
    }
    const float2 before = pick(o.p, j);
    put(o.p, j, st.p);
    put(o.q, j, st.po);
    c.xy[li] = st.p;
    c.vel[li] = st.vel;
    // (an upper bound will do: the root's last bits do not matter)
    const float tx = (st.p.x - before.x) - w.drift.x, ty = (st.p.y - before.y) - w.drift.y;
    const float travel = pick(o.travel, j) + 1.0001f * __builtin_amdgcn_sqrtf(tx * tx + ty * ty);
    put(o.travel, j, travel);
    if (finitef(st.p.x) && finitef(st.p.y) && !(travel <= w.skin) && ((o.nl >> (4u * j)) & 15u) != kOut) {
        const uint32_t u = atomicAdd(&c.out->n, 1u);
        if (u < kOutMax) {
            c.out->id[u] = (uint16_t)li;
            o.nl |= kOut << (4u * j);
        }
    }
}

// The bodies filed by cell (rec, c.cnt) and, unless w.grid, everyone's list of the bodies it could
// touch until one of the two has travelled w.skin.
static __device__ __forceinline__ void build_lists(Ctx& c, Own& o, Walk& w, const DiffArgs& a, const DiffWorld& W) {
    const uint32_t tid = thread_index();
    const uint32_t per = per_thread(W);
    if (w.grid == 0 || w.grid % kFitEvery == 0) {
        LdsFit f;
        f.init();
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j)
            if (tid + j * kDiffThreads < W.nb) {
                f.point(o.p[j].x, o.p[j].y);
                if (!(o.fl[j] & BF_STATIC)) f.extra(o.p[j].x - o.q[j].x, o.p[j].y - o.q[j].y);
            }
        lds_fit<kDiffThreads>(f, 2.004f * (W.rmax + (w.grid ? 0.0f : w.skin)), kDiffCells, c.red, c.grid);
    }
    const LdsGrid g = lds_grid_uniform(*c.grid);
    w.drift = make_float2(g.ex, g.ey);
    w.tested = 0;
    for (uint32_t i = tid; i <= g.ncells; i += kDiffThreads) c.cnt[i] = 0u;
    if (tid == 0) c.out->n = 0;
    __syncthreads();
    uint32_t key[PER] = {}, at[PER] = {};
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j)
        if (tid + j * kDiffThreads < W.nb) {
            key[j] = lds_cell(g, o.p[j].x, o.p[j].y);
            at[j] = atomicAdd(&c.cnt[key[j]], 1u);
        }
    __syncthreads();
    lds_scan<kDiffThreads, kScanItems>(c.cnt, g.ncells + 1u, c.red);
    c.rec = w.grid ? reinterpret_cast<float4*>(c.lists) : c.force;
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        const uint32_t li = tid + j * kDiffThreads;
        if (li >= W.nb) continue;
        at[j] += c.cnt[key[j]];
        c.rec[at[j]] = make_float4(o.p[j].x, o.p[j].y, c.rad[li], __uint_as_float(li));
        o.travel[j] = 0.0f;
    }
    __syncthreads();
    if (w.grid) return;
    for (uint32_t tries = 1;; ++tries) {
        o.nl = 0;
#pragma unroll 1
        for (uint32_t j = 0; j < per; ++j) {
            const uint32_t li = tid + j * kDiffThreads;
            const float2 xy = pick(o.p, j);
            if (li >= W.nb || !finitef(xy.x) || !finitef(xy.y)) continue;
            const float r = c.rad[li];
            const float reach = r + 2.0f * w.skin + (1e-4f * (r + W.rmax + 2.0f * w.skin) + 1e-5f);
            const LdsRows l = lds_rows(g, c.cnt, true, xy, reach + W.rmax);
            const uint64_t near = lds_near(l, c.rec, [&](uint32_t, const float4& b) {
                const float dx = xy.x - b.x, dy = xy.y - b.y, rs = reach + b.z;
                return !((__float_as_uint(b.w) == li) | (dx * dx + dy * dy > rs * rs));
            });
            const uint32_t n = (uint32_t)__popcll(near);
            if (l.flat && n <= kListCap) {
                uint32_t i = 0;
                for (uint64_t m = near; m != 0; m &= m - 1, ++i)
                    c.lists[i >> 2][li][i & 3u] =
                        (uint16_t)__float_as_uint(c.rec[l.slot((uint32_t)__builtin_ctzll(m))].w);
                for (; (i & 3u) != 0u; ++i) c.lists[i >> 2][li][i & 3u] = (uint16_t)li;  // (whole groups are read)
                o.nl |= n << (4u * j);
            } else {
                const uint32_t u = atomicAdd(&c.out->n, 1u);
                if (u < kOutMax) c.out->id[u] = (uint16_t)li;
                o.nl |= kOut << (4u * j);
            }
        }
        static_assert(kListCap < kOut && kListCap <= 8, "four bits; the mask below");
        __syncthreads();
        if (c.out->n <= kOutMax) break;
        __syncthreads();
        if (tries == kListTries) {  // the world is too dense for lists: file it every substep
            w.grid = kGridHold;
            w.skin = kSkin * 2.0f * W.rmax;
            c.rec = reinterpret_cast<float4*>(c.lists);
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                const uint32_t li = tid + j * kDiffThreads;
                if (li < W.nb) c.rec[at[j]] = make_float4(o.p[j].x, o.p[j].y, c.rad[li], __uint_as_float(li));
            }
            if (tid == 0) c.out->n = 0;
            __syncthreads();
            break;
        }
        w.skin *= 0.5f;
        if (tid == 0) c.out->n = 0;
        __syncthreads();
    }
}

// Mark phase of the lists: the pairs within reach go into the queue.  Returns body 0's and body
// 1's pairs, first | n << 16 (n kNoRoom: worked out by the body's thread).
static constexpr uint32_t kNoRoom = 0xFFFFu;
static __device__ __forceinline__ void mark_lists(Ctx& c, const Own& o, const DiffWorld& W, uint32_t par,
                                           uint32_t (&pr)[PER]) {
    const uint32_t tid = thread_index();
    const uint32_t per = per_thread(W);
    const uint32_t nout = (uint32_t)__builtin_amdgcn_readfirstlane((int)c.out->n);
    uint32_t* count = &c.out->pairs[par];
    auto within = [&](float2 p, float r, float2 b, float rb) {
        const float dx = p.x - b.x, dy = p.y - b.y, rs = r + rb;
        return !(dx * dx + dy * dy > (rs * rs) * 1.00000095367431640625f);
    };
    auto near = [&](float2 p, float r, uint32_t lj) { return within(p, r, c.xy[lj], c.rad[lj]); };
    // the outliers, one a lane, read from there by every lane
    const uint32_t lane = tid & (BG_WAVE - 1);
    const uint32_t out_id = lane < nout ? c.out->id[lane] : 0u;
    const float2 out_p = c.xy[out_id];
    const float out_r = c.rad[out_id];
    auto of_lane = [](float v, uint32_t u) {
        return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), (int)u));
    };
#pragma unroll 1
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t li = tid + j * kDiffThreads;
        uint32_t marked = 0;
        const uint32_t nl = (o.nl >> (4u * j)) & 15u;
        const float2 p = pick(o.p, j);
        if (li < W.nb && finitef(p.x) && finitef(p.y)) {
            const float r = c.rad[li];
            const uint32_t n = nl != kOut ? nl : 0u;
            uint2 l[kListCap / 4];
#pragma unroll
            for (uint32_t f = 0; f < kListCap / 4; ++f) {
                l[f] = make_uint2(0u, 0u);
                if (4 * f >= n) continue;
                l[f] = *(const uint2*)c.lists[f][li];
                marked |= ((near(p, r, l[f].x & 0xFFFFu) ? 1u : 0u) | (near(p, r, l[f].x >> 16) ? 2u : 0u) |
                           (near(p, r, l[f].y & 0xFFFFu) ? 4u : 0u) | (near(p, r, l[f].y >> 16) ? 8u : 0u))
                          << (4 * f);
            }
            marked &= (1u << n) - 1u;
            // (a body outside the lists leaves its pairs with the others to them)
            for (uint32_t u = 0; u < nout; ++u) {
                const uint32_t lj = (uint32_t)__builtin_amdgcn_readlane((int)out_id, (int)u);
                if (lj == li || !within(p, r, make_float2(of_lane(out_p.x, u), of_lane(out_p.y, u)), of_lane(out_r, u)))
                    continue;
                bool listed = false;  // (then its entry has been marked)
#pragma unroll
                for (uint32_t f = 0; f < kListCap / 4; ++f) {
                    listed |= 4 * f < n && (l[f].x & 0xFFFFu) == lj;
                    listed |= 4 * f + 1 < n && (l[f].x >> 16) == lj;
                    listed |= 4 * f + 2 < n && (l[f].y & 0xFFFFu) == lj;
                    listed |= 4 * f + 3 < n && (l[f].y >> 16) == lj;
                }
                if (!listed && nl != kOut) marked |= 1u << (kListCap + u);
                // and the pair from the other's side
                const uint32_t k = atomicAdd(&c.out->count[par][u], 1u);
                if (k < kOutPairs) c.entries[kPairs + u * kOutPairs + k] = (lj << 16) | li;
            }
        }
        const LdsPairs q = lds_queue<kPairs>(marked, li, c.entries, count, [&](uint32_t i) {
            return i < kListCap ? (uint32_t)c.lists[i >> 2][li][i & 3u] : (uint32_t)c.out->id[i - kListCap];
        });
        put(pr, j, q.first | (q.direct ? kNoRoom : q.n) << 16);
    }
    static_assert(kListCap + kOutMax <= 32, "the mask");
}

// The contacts of the bodies still to do (bit j of `pending`), as many of them at a time as the
// queue has room for: a world of thousands of pairs, or one without lists.  (A thread doing all of
// its body's, candidate by candidate, leaves the wave to its busiest: 4 worlds of 2,048 bodies
// thrown on eight times their area's worth, 10 steps: 28.6 ms, 88.0 that way.)
//
// Bound by the walks over the candidates, so one walk both counts a body's partners and keeps the
// last kKept of them, and only a body of more is walked again to enter them.  A thread's two bodies
// are done one after the other, written out twice (in a loop the state in flight costs 10%).  Against
// two walks of every body and a loop, forward, us: 8 worlds of 700 with their positions scaled by
// 0.4 1,850 -> 1,160, of 1,500 5,420 -> 3,260, of 2,048 7,310 -> 3,790; by 0.15, of 2,048 29,900 -> 24,400.
template <class Contact, class Finish>
static __device__ __forceinline__ void queue_rounds(Ctx& c, const Own& o, const DiffWorld& W, bool lists, uint32_t nout,
                                                    uint32_t pending, Contact&& contact, Finish&& finish) {
    const uint32_t tid = thread_index();
    const uint32_t per = per_thread(W);
    // f(partner) for the candidates of body j within reach
    auto partners = [&](uint32_t j, auto&& f) {
        const uint32_t li = tid + j * kDiffThreads;
        const float2 p = pick(o.p, j);
        const float r = c.rad[li];
        auto test = [&](uint32_t lj, float2 b, float rb) {
            const float dx = p.x - b.x, dy = p.y - b.y, rs = r + rb;
            if ((lj != li) & !(dx * dx + dy * dy > (rs * rs) * 1.00000095367431640625f)) f(lj);
        };
        const uint32_t n = (o.nl >> (4u * j)) & 15u;
        if (!lists) {
            const LdsGrid g = lds_grid_uniform(*c.grid);
            const LdsRect q = lds_rect(g, p.x, p.y, r + W.rmax);
            for (int32_t cy = q.cy0; cy <= q.cy1; ++cy) {
                const uint32_t row = (uint32_t)cy * (uint32_t)g.nx;
                const uint32_t t1 = c.cnt[row + (uint32_t)q.cx1 + 1u];
                for (uint32_t t = c.cnt[row + (uint32_t)q.cx0]; t < t1; t += 4) {
                    float4 b[4];
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) b[u] = c.rec[t + u];
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u)
                        if (t + u < t1) test(__float_as_uint(b[u].w), make_float2(b[u].x, b[u].y), b[u].z);
                }
            }
            static_assert(kLdsRecPad >= 3, "reads past the last record");
        } else {
            for (uint32_t i = 0; i < n; ++i) {
                const uint32_t lj = c.lists[i >> 2][li][i & 3u];
                test(lj, c.xy[lj], c.rad[lj]);
            }
            for (uint32_t u = 0; u < nout; ++u) {
                const uint32_t lj = c.out->id[u];
                bool listed = false;
                for (uint32_t i = 0; i < n; ++i) listed |= c.lists[i >> 2][li][i & 3u] == lj;
                if (!listed) test(lj, c.xy[lj], c.rad[lj]);
            }
        }
    };
    // The same by the whole wave for a body outside the lists, which tests everyone: f(hit, lj, the hits'
    // lanes) for 64 candidates at a time.  (Its lane alone took some 50 us a substep of a world of 700: 8 of
    // them scaled by 0.55, a little too dense for lists, 1,190 us forward for 4 steps, 745 so.)
    const uint32_t lane = tid & (BG_WAVE - 1);
    auto everyone = [&](uint32_t li, auto&& f) {
        const float2 p = c.xy[li];
        const float r = c.rad[li];
        for (uint32_t base = 0; base < W.nb; base += BG_WAVE) {
            const uint32_t lj = base + lane;
            bool hit = false;
            if (lj < W.nb) {
                const float2 b = c.xy[lj];
                const float dx = p.x - b.x, dy = p.y - b.y, rs = r + c.rad[lj];
                hit = (lj != li) & !(dx * dx + dy * dy > (rs * rs) * 1.00000095367431640625f);
            }
            f(hit, lj, __ballot(hit));
        }
    };
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        if (j >= per) break;
        bool todo = ((pending >> j) & 1u) != 0u;
        const uint32_t own = (tid + j * kDiffThreads) << 16;
        const bool all = todo && lists && ((o.nl >> (4u * j)) & 15u) == kOut;
        uint32_t need = 0;
        uint32_t kept[kKept / 2] = {};  // the last kKept partners found, 16 bits each
        for (uint64_t m = __ballot(all); m; m &= m - 1) {
            const int l = __builtin_ctzll(m);
            uint32_t n = 0;
            everyone((uint32_t)__builtin_amdgcn_readlane((int)own, l) >> 16,
                     [&](bool, uint32_t, uint64_t hits) { n += (uint32_t)__popcll(hits); });
            if (lane == (uint32_t)l) need = n;
        }
        if (todo && !all)
            partners(j, [&](uint32_t lj) {
                ++need;
#pragma unroll
                for (uint32_t k = kKept / 2 - 1; k > 0; --k) kept[k] = kept[k] << 16 | kept[k - 1] >> 16;
                kept[0] = kept[0] << 16 | lj;
            });
        const bool never = need > kPairs;  // fits the queue
        for (;;) {  // (the first body in line fits, so every round does some)
            __syncthreads();
            if (tid == 0) c.out->round = c.out->more = 0;
            __syncthreads();
            const uint32_t n = todo && !never ? need : 0u;
            const uint32_t incl = wave_prefix(n, 0u, AddU32());
            const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, BG_WAVE - 1);
            uint32_t first = 0;
            if (total > 0 && (tid & (BG_WAVE - 1)) == 0) first = atomicAdd(&c.out->round, total);
            first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first) + incl - n;
            const bool placed = todo && (never || first + n <= kPairs);
            for (uint64_t m = __ballot(all && placed && !never); m; m &= m - 1) {
                const int l = __builtin_ctzll(m);
                const uint32_t body = (uint32_t)__builtin_amdgcn_readlane((int)own, l);
                uint32_t e = (uint32_t)__builtin_amdgcn_readlane((int)first, l);
                const uint32_t e1 = e + (uint32_t)__builtin_amdgcn_readlane((int)need, l);
                const float2 range = make_float2(__uint_as_float(e), __uint_as_float(e1));
                everyone(body >> 16, [&](bool hit, uint32_t lj, uint64_t hits) {
                    if (hit) {
                        const uint32_t at = e + (uint32_t)__popcll(hits & lanemask_lt());
                        c.entries[at] = body | lj;
                        c.res[at] = range;
                    }
                    e += (uint32_t)__popcll(hits);
                });
            }
            if (placed && !never && !all) {
                uint32_t e = first;
                const float2 range = make_float2(__uint_as_float(first), __uint_as_float(first + n));
                auto enter = [&](uint32_t lj) {
                    c.entries[e] = own | lj;
                    c.res[e++] = range;
                };
                if (n <= kKept) {
                    while (e < first + n) {
                        enter(kept[0] & 0xFFFFu);
#pragma unroll
                        for (uint32_t k = 0; k + 1 < kKept / 2; ++k) kept[k] = kept[k] >> 16 | kept[k + 1] << 16;
                        kept[kKept / 2 - 1] >>= 16;
                    }
                } else {
                    partners(j, enter);
                }
            } else if (todo && !placed) {
                for (uint32_t e = first; e < kPairs; ++e) c.entries[e] = kNoPair;
            }
            __syncthreads();
            // a pair's correction, and its place in its body's ascending order (dozens of partners would
            // take a thread by itself long to sort)
            uint32_t to[2], key[2];
            float2 k[2];
            static_assert(kPairs <= 2 * kDiffThreads, "the two");
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
                const uint32_t e = tid + i * kDiffThreads;
                to[i] = kNoPair;
                if (e >= min(c.out->round, kPairs)) continue;
                const uint32_t pair = c.entries[e];
                if (pair == kNoPair) continue;
                to[i] = __float_as_uint(c.res[e].x);
                const uint32_t end = __float_as_uint(c.res[e].y);
#pragma unroll 4
                for (uint32_t f = __float_as_uint(c.res[e].x); f < end; ++f) to[i] += c.entries[f] < pair ? 1u : 0u;
                const LdsContact ct = contact(pair >> 16, pair & 0xFFFFu);
                key[i] = ct.hit ? pair & 0xFFFFu : kNoPair;
                k[i] = ct.c;
            }
            __syncthreads();
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i)
                if (to[i] != kNoPair) {
                    c.entries[to[i]] = key[i];
                    c.res[to[i]] = k[i];
                }
            __syncthreads();
            if (placed) finish(j, first, never ? kNoRoom : need, !never);
            todo = todo && !placed;
            if (todo) c.out->more = 1;
            __syncthreads();
            if (__builtin_amdgcn_readfirstlane((int)c.out->more) == 0) break;
        }
    }
}

// One forward substep of the world (`n` counts this launch's substeps); with
// REC, records the snapshot, contact partners, velocities (damped springs) and
// joint-stage positions (joints) at tape slot `slot`.
template <bool REC>
static __device__ __forceinline__ void substep_forward(Ctx& c, Own& o, Walk& w, const DiffArgs& a, const DiffWorld& W,
                                                uint32_t gsub, uint32_t n, uint32_t slot) {
    const uint32_t tid = thread_index();
    const bool springs_lds = lds_springs(W);
    const bool joints = W.njg > 0;
    const uint32_t per = per_thread(W), par = n & 1u;
    if (a.collisions && w.build) build_lists(c, o, w, a, W);
    const bool lists = a.collisions && w.grid == 0;
    if (springs_lds) {
        own_springs(o, a, W, [&](uint32_t t, uint32_t ia, uint32_t ib, float rest, float k, float cc) {
            const float2 f = spring_force(c.xy[ia], c.xy[ib], c.vel[ia], c.vel[ib], rest, k, cc);
            const float ma = c.mass[ia], mb = c.mass[ib];
            c.force[t] = make_float4(f.x / ma, f.y / ma, (-f.x) / mb, (-f.y) / mb);
        });
    } else {
        // too many springs for LDS: each body sums its own into its entry of `force`
        for (uint32_t j = 0; j < per; ++j) {
            const uint32_t li = tid + j * kDiffThreads, gi = W.b0 + li;
            if (li >= W.nb) continue;
            float2 ac = gsub == 0 ? a.acc0[gi] : make_float2(0.0f, 0.0f);
            ac.x = ac.x + a.gx * c.gmod[li];
            ac.y = ac.y + a.gy * c.gmod[li];
            const float m = c.mass[li];
            for (uint32_t e = a.inc_start[gi]; e < a.inc_start[gi + 1]; ++e) {
                const uint32_t s = a.inc_list[e];
                const uint32_t ia = (uint32_t)a.sp_a[s] - W.b0, ib = (uint32_t)a.sp_b[s] - W.b0;
                const float2 f =
                    spring_force(c.xy[ia], c.xy[ib], c.vel[ia], c.vel[ib], a.sp_rest[s], a.sp_k[s], a.sp_c[s]);
                ac.x = ac.x + (li == ia ? f.x : -f.x) / m;
                ac.y = ac.y + (li == ia ? f.y : -f.y) / m;
            }
            c.force[li] = make_float4(ac.x, ac.y, 0.0f, 0.0f);
        }
    }
    // contacts against the snapshot (physics.rs:241-317)
    uint32_t pr[PER] = {}, nout = 0;
    bool crowd = a.collisions && !lists;
    auto contact = [&](uint32_t li, uint32_t lj) {
        const float2 p = c.xy[li], b = c.xy[lj];
        return lds_correction(make_float4(p.x, p.y, c.rad[li], 0.0f), make_float4(b.x, b.y, c.rad[lj], 0.0f),
                              c.mass[li], c.mass[lj], li > lj, false);
    };
    if (lists) {
        mark_lists(c, o, W, par, pr);
        __syncthreads();
        // (read here: past the next barrier somebody may already be at the end of the substep)
        nout = (uint32_t)__builtin_amdgcn_readfirstlane((int)c.out->n);
        crowd = c.out->pairs[par] > kPairs;
        crowd |= __any((tid & (BG_WAVE - 1)) < nout && c.out->count[par][tid & (kOutMax - 1)] > kOutPairs) != 0;
        const uint32_t queued = min(c.out->pairs[par], kPairs);
        const uint32_t total = queued + nout * kOutPairs;
        for (uint32_t i = tid; i < total; i += kDiffThreads) {
            uint32_t e = i;
            if (i >= queued) {
                const uint32_t u = (i - queued) / kOutPairs, k = (i - queued) % kOutPairs;
                if (k >= c.out->count[par][u]) continue;
                e = kPairs + i - queued;
            }
            const uint32_t pair = c.entries[e];
            if (pair == kNoPair) continue;
            const LdsContact k = contact(pair >> 16, pair & 0xFFFFu);
            c.entries[e] = k.hit ? pair & 0xFFFFu : kNoPair;
            c.res[e] = k.c;
        }
    }
    __syncthreads();
    // A body's corrections, ascending partner index, from `count` entries of the queue (kNoRoom: from
    // all bodies, one after the other); the tape takes the first kDiffTapeNbr - 1 partners.
    float2 sums[PER] = {};
    auto finish = [&](uint32_t j, uint32_t first, uint32_t count, bool sorted) {
        const uint32_t li = tid + j * kDiffThreads;
        float2 pn = pick(o.p, j);
        uint32_t w0 = 0xFFFF0000u, w1 = 0xFFFFFFFFu, w2 = 0xFFFFFFFFu, w3 = 0xFFFFFFFFu, found = 0;
        auto add = [&](uint32_t t, uint32_t lj, float2 k) {  // partner number t
            pn.x = pn.x + k.x;
            pn.y = pn.y + k.y;
            if (!REC) return;
            const uint32_t keep = t & 1u ? 0xFFFF0000u : 0xFFFFu, put_ = t & 1u ? lj : lj << 16;
            if (t < 1) w0 = (w0 & keep) | put_;
            else if (t < 3) w1 = (w1 & keep) | put_;
            else if (t < 5) w2 = (w2 & keep) | put_;
            else if (t < 7) w3 = (w3 & keep) | put_;
        };
        static_assert(kDiffTapeNbr == 8, "four words: the count and seven partners");
        if (sorted) {
            for (uint32_t e = first; e < first + count; ++e)
                if (c.entries[e] != kNoPair) add(found++, c.entries[e], c.res[e]);
        } else if (count != kNoRoom) {
            found = lds_sum({first, count, false}, c.entries, c.res, add);
        } else {
            for (uint32_t lj = 0; lj < W.nb; ++lj) {
                const LdsContact k = contact(li, lj);
                if (lj != li && k.hit) add(found++, lj, k.c);
            }
        }
        if (REC && a.collisions) {
            w0 |= found < 0xFFFFu ? found : 0xFFFFu;
            reinterpret_cast<uint4*>(a.tape_nbr)[(size_t)slot * a.nb_total + W.b0 + li] = make_uint4(w0, w1, w2, w3);
        }
        put(sums, j, pn);
    };
    uint32_t pending = 0;  // bit j: body j's contacts are still to do
#pragma unroll 1
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t li = tid + j * kDiffThreads;
        if (li >= W.nb) continue;
        const float2 xy = pick(o.p, j);
        if (REC) a.tape_s[(size_t)slot * a.nb_total + W.b0 + li] = xy;
        uint32_t first = 0, count = 0;
        if (lists) {
            first = pick(pr, j) & 0xFFFFu;
            count = pick(pr, j) >> 16;
            if (((o.nl >> (4u * j)) & 15u) == kOut)
                for (uint32_t u = 0; u < nout; ++u)
                    if (c.out->id[u] == li) {
                        first = kPairs + u * kOutPairs;
                        count = c.out->count[par][u] <= kOutPairs ? c.out->count[par][u] : kNoRoom;
                    }
        } else if (a.collisions && finitef(xy.x) && finitef(xy.y)) {
            count = kNoRoom;
        }
        if (count == kNoRoom)
            pending |= 1u << j;
        else
            finish(j, first, count, false);
    }
    // (The hint keeps the rounds' state from taking registers that two bodies a thread need in every
    // substep: 256 worlds of 2,048 over 50 steps 4.83 ms without it, 4.76 with.  With one body a thread
    // it costs 96 worlds of 700 a hundredth.)
    if (PER == 1 ? crowd : __builtin_expect(crowd, 0)) queue_rounds(c, o, W, lists, nout, pending, contact, finish);
    if (tid == 0) c.out->pairs[par ^ 1u] = 0;
    if (tid < kOutMax) c.out->count[par ^ 1u][tid] = 0;
    // From here to the end of the substep a thread touches the positions and velocities of its
    // own bodies only, so it may rewrite them.
#pragma unroll 1
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t li = tid + j * kDiffThreads, gi = W.b0 + li;
        if (li >= W.nb) continue;
        const float2 pn = pick(sums, j);
        if (REC && a.tape_v) a.tape_v[(size_t)slot * a.nb_total + gi] = c.vel[li];
        // gravity + springs (physics.rs:369-375, springs.rs:25-47), ascending spring index
        float2 ac = make_float2(0.0f, 0.0f);
        if (springs_lds) {
            if (!(pick(o.fl, j) & BF_STATIC)) {
                if (gsub == 0) ac = a.acc0[gi];
                ac.x = ac.x + a.gx * c.gmod[li];
                ac.y = ac.y + a.gy * c.gmod[li];
                for_springs(o, j, a, W, [&](uint32_t e) {
                    const float2 f = reinterpret_cast<const float2*>(c.force)[e];
                    ac.x = ac.x + f.x;
                    ac.y = ac.y + f.y;
                });
            }
        } else {
            ac = make_float2(c.force[li].x, c.force[li].y);
        }
        if (joints) {
            c.vel[li] = pn;
            c.xy[li] = ac;
        } else {
            verlet(c, o, w, a, W, gsub, j, pn, ac);
        }
    }
    __syncthreads();
    // fixed joints, positions (physics.rs:424-460), on the velocities' memory
    if (joints) {
        if (joints_staged(W))
            joint_sweep<REC, true>(c, c.vel, a, W, slot);
        else
            joint_sweep<REC, false>(c, c.vel, a, W, slot);
        __syncthreads();
        for (uint32_t j = 0; j < per; ++j) {
            const uint32_t li = tid + j * kDiffThreads;
            if (li < W.nb) verlet(c, o, w, a, W, gsub, j, c.vel[li], c.xy[li]);
        }
        __syncthreads();
    }
    if (w.grid) --w.grid;
    nout = (uint32_t)__builtin_amdgcn_readfirstlane((int)c.out->n);
    w.tested += nout;
    w.build = !lists || nout > kOutMax || w.tested > kTested;
}

// One tape slot of a thread's bodies (the contact partners are loaded by the substep itself,
// which needs them late).
struct Tape {
    float2 s[PER], v[PER];
    float2 axis;  // of one of a staged world's solves
};

static __device__ __forceinline__ void load_tape(Tape& t, const DiffArgs& a, const DiffWorld& W, uint32_t k) {
    const uint32_t tid = thread_index();
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        const uint32_t li = tid + j * kDiffThreads;
        if (li >= W.nb) continue;
        const size_t i = (size_t)k * a.nb_total + W.b0 + li;
        t.s[j] = a.tape_s[i];
        if (a.tape_v) t.v[j] = a.tape_v[i];
    }
    if (joints_staged(W) && tid < W.nje) t.axis = a.tape_axis[(size_t)k * a.n_solves + W.je0 + tid];
}

// Terms of one spring's adjoint: d loss / d (p_b - p_a) (kx, ky), d loss /
// d (v_a - v_b) (rvx, rvy) and d loss / d stiffness.
struct SpringAdj {
    float kx, ky, rvx, rvy, gk;
};
static __device__ __forceinline__ SpringAdj spring_adjoint(const Ctx& c, uint32_t ia, uint32_t ib, float rest, float kk, float cc) {
    SpringAdj r;
    const float4 pa = c.rec[ia], pb = c.rec[ib];
    const float dx = pb.x - pa.x, dy = pb.y - pa.y;
    const float L = sqrtf(dx * dx + dy * dy);
    const float ux = dx / L, uy = dy / L;
    const float2 la = c.lam_am[ia], lb = c.lam_am[ib];
    const float lfx = la.x - lb.x, lfy = la.y - lb.y;
    const float uf = ux * lfx + uy * lfy;
    const float t = kk * (1.0f - rest / L);
    r.kx = t * (lfx - ux * uf) + kk * ux * uf;
    r.ky = t * (lfy - uy * uf) + kk * uy * uf;
    r.rvx = r.rvy = 0.0f;
    if (cc != 0.0f) {
        const float2 va = c.vel[ia], vb = c.vel[ib];
        const float vx = va.x - vb.x, vy = va.y - vb.y;
        const float dot = vx * ux + vy * uy;
        const float wl = ux * ux * lfx + uy * uy * lfy;
        // d loss / d u of -c dot (u_x^2, u_y^2), then through du/dd = (I - u u^T)/L
        const float gux = -cc * (vx * wl + 2.0f * dot * ux * lfx);
        const float guy = -cc * (vy * wl + 2.0f * dot * uy * lfy);
        const float gu = ux * gux + uy * guy;
        r.kx += (gux - ux * gu) / L;
        r.ky += (guy - uy * gu) / L;
        r.rvx = -cc * wl * ux;
        r.rvy = -cc * wl * uy;
    }
    r.gk = (L - rest) * uf;
    return r;
}

// Adjoint of substep `gsub`, tape slot k, whose positions are in `t`.  In: lp,
// lq, lv = d loss / d (position, position_old, calculated_velocity) after the
// substep.  Out: the same before it; gv += d loss / d velocity_request at the
// substep that consumes it; gk: the stiffness gradient of the thread's first
// spring.  With `more`, `t` leaves with slot k - 1 on its way.
static __device__ __forceinline__ void substep_reverse(Ctx& c, const Own& o, const DiffArgs& a, const DiffWorld& W,
                                                uint32_t gsub, uint32_t k, bool more, Tape& t, float2 (&lp)[PER],
                                                float2 (&lq)[PER], float2 (&lv)[PER], float2 (&gv)[PER], float& gk) {
    const uint32_t tid = thread_index();
    const float h = a.h;
    const bool joints = W.njg > 0;
    const bool springs_lds = lds_springs(W);
    const uint32_t per = per_thread(W);
    // per spring (kx, ky) and, with damping, (rvx, rvy): the memory of a cell table and of the
    // forward's positions is free
    float2* skx = c.spring_k;
    float2* srv = c.spring_v;
    uint4 nbr[PER];
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        const uint32_t li = tid + j * kDiffThreads;
        nbr[j] = make_uint4(0u, 0u, 0u, 0u);
        if (li >= W.nb) continue;
        if (a.collisions)
            nbr[j] = reinterpret_cast<const uint4*>(a.tape_nbr)[(size_t)k * a.nb_total + W.b0 + li];
        const float m = c.mass[li];
        c.rec[li] = make_float4(t.s[j].x, t.s[j].y, c.rad[li], m);
        if (a.tape_v) c.vel[li] = t.v[j];
        float2 lam_a = make_float2(0.0f, 0.0f), lpp, lqin = make_float2(0.0f, 0.0f);
        if (o.fl[j] & BF_STATIC) {  // p'' = p', q'' = p', v'' = 0
            lpp = make_float2(lp[j].x + lq[j].x, lp[j].y + lq[j].y);
        } else {
            // dx = (p' - q) r; p'' = p' + dx + a h^2, q'' = p', v'' = dx / h
            const float ratio = ((int32_t)li == W.first_dyn && gsub == 0) ? h / W.old_dt0 : h / h;
            const float ldx = lp[j].x + lv[j].x / h, ldy = lp[j].y + lv[j].y / h;
            if (gsub == 0 && (o.fl[j] & BF_HAS_VREQ)) {  // q = p' - vreq h: dx = vreq h r
                lpp = make_float2(lp[j].x + lq[j].x, lp[j].y + lq[j].y);
                gv[j].x += h * ratio * ldx;
                gv[j].y += h * ratio * ldy;
            } else {
                lpp = make_float2((lp[j].x + lq[j].x) + ratio * ldx, (lp[j].y + lq[j].y) + ratio * ldy);
                lqin = make_float2(-ratio * ldx, -ratio * ldy);
            }
            lam_a = make_float2(h * h * lp[j].x / m, h * h * lp[j].y / m);
        }
        lq[j] = lqin;
        c.lam_pp[li] = lpp;
        c.lam_am[li] = lam_a;
    }
    if (joints && joints_staged(W) && tid < W.nje) c.axes[tid] = t.axis;
    if (more) load_tape(t, a, W, k - 1);
    __syncthreads();
    if (joints) {
        if (joints_staged(W))
            joint_sweep_reverse<true>(c, c.lam_pp, a, W, k);
        else
            joint_sweep_reverse<false>(c, c.lam_pp, a, W, k);
        __syncthreads();
    }
    if (springs_lds && W.ns > 0) {
        own_springs(o, a, W, [&](uint32_t s, uint32_t ia, uint32_t ib, float rest, float kk, float cc) {
            const SpringAdj r = spring_adjoint(c, ia, ib, rest, kk, cc);
            skx[s] = make_float2(r.kx, r.ky);
            if (a.tape_v) srv[s] = make_float2(r.rvx, r.rvy);
            if (s < kDiffThreads)
                gk += r.gk;
            else
                a.grad_k[W.s0 + s] += r.gk;
        });
        __syncthreads();
    }
#pragma unroll 1
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t li = tid + j * kDiffThreads, gi = W.b0 + li;
        if (li >= W.nb) continue;
        const float4 si = c.rec[li];
        const float2 lpp = c.lam_pp[li];
        float2 ls = make_float2(0.0f, 0.0f), lvin = make_float2(0.0f, 0.0f);
        // contacts, pair set of the forward substep
        if (a.collisions && finitef(si.x) && finitef(si.y)) {
            auto pair = [&](uint32_t lj) {
                const float4 sj = c.rec[lj];
                const float ax = si.x - sj.x, ay = si.y - sj.y;
                const float d = sqrtf(ax * ax + ay * ay);
                if (!(d >= 1e-6f)) return;  // push-out branch: held constant
                const float rs = si.z + sj.z;
                const float wi = sj.w / (si.w + sj.w), wj = si.w / (si.w + sj.w);
                const float2 lj2 = c.lam_pp[lj];
                const float mux = wi * lpp.x - wj * lj2.x, muy = wi * lpp.y - wj * lj2.y;
                const float nx = ax / d, ny = ay / d;
                const float nm = nx * mux + ny * muy;
                const float f = rs / d;
                ls.x += f * (mux - nx * nm) - mux;
                ls.y += f * (muy - ny * nm) - muy;
            };
            uint4 words = nbr[0];
            if constexpr (PER == 2) words = make_uint4(j ? nbr[1].x : words.x, j ? nbr[1].y : words.y,
                                                       j ? nbr[1].z : words.z, j ? nbr[1].w : words.w);
            uint32_t w0 = words.x, w1 = words.y, w2 = words.z, w3 = words.w;
            const uint32_t n = w0 & 0xFFFFu;
            if (n < kDiffTapeNbr) {
                for (uint32_t i = 0; i < n; ++i) {  // shift the next partner down
                    w0 = (w0 >> 16) | (w1 << 16);
                    w1 = (w1 >> 16) | (w2 << 16);
                    w2 = (w2 >> 16) | (w3 << 16);
                    w3 >>= 16;
                    pair(w0 & 0xFFFFu);
                }
            } else {  // more partners than the tape holds: the same predicate over the world
                for (uint32_t lj = 0; lj < W.nb; ++lj) {
                    if (lj == li) continue;
                    const float4 sb = c.rec[lj];
                    const bool isA = li > lj;
                    const float ax = isA ? si.x - sb.x : sb.x - si.x;
                    const float ay = isA ? si.y - sb.y : sb.y - si.y;
                    const float rs = si.z + sb.z;
                    const float dot = ax * ax + ay * ay;
                    if (dot > (rs * rs) * 1.00000095367431640625f) continue;
                    if (!(sqrtf(dot) < rs)) continue;
                    pair(lj);
                }
            }
        }
        // springs
        auto add = [&](bool is_a, float kx, float ky, float rvx, float rvy) {
            if (is_a) {
                ls.x -= kx;
                ls.y -= ky;
                lvin.x += rvx;
                lvin.y += rvy;
            } else {
                ls.x += kx;
                ls.y += ky;
                lvin.x -= rvx;
                lvin.y -= rvy;
            }
        };
        if (springs_lds) {
            for_springs(o, j, a, W, [&](uint32_t e) {
                const float2 kxy = skx[e >> 1];
                const float2 rv = a.tape_v ? srv[e >> 1] : make_float2(0.0f, 0.0f);
                add((e & 1u) == 0u, kxy.x, kxy.y, rv.x, rv.y);
            });
        } else {
            for (uint32_t e = a.inc_start[gi]; e < a.inc_start[gi + 1]; ++e) {
                const uint32_t s = a.inc_list[e];
                const uint32_t ia = (uint32_t)a.sp_a[s] - W.b0, ib = (uint32_t)a.sp_b[s] - W.b0;
                const SpringAdj r = spring_adjoint(c, ia, ib, a.sp_rest[s], a.sp_k[s], a.sp_c[s]);
                add(li == ia, r.kx, r.ky, r.rvx, r.rvy);
                if (li == ia) a.grad_k[s] += r.gk;
            }
        }
        put(lp, j, make_float2(lpp.x + ls.x, lpp.y + ls.y));
        put(lv, j, lvin);
    }
    __syncthreads();  // snapshot and adjoint vectors are rewritten by the next substep
}

// Centroid of the world's positions (f64 sums) by the block.
static __device__ double2 block_centroid(Ctx& c, const Own& o, const DiffWorld& W) {
    double sx = 0.0, sy = 0.0;
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j)
        if (threadIdx.x + j * kDiffThreads < W.nb) {
            sx += (double)o.p[j].x;
            sy += (double)o.p[j].y;
        }
    for (int off = 32; off > 0; off >>= 1) {
        sx += __shfl_xor(sx, off, BG_WAVE);
        sy += __shfl_xor(sy, off, BG_WAVE);
    }
    const int lane = threadIdx.x & (BG_WAVE - 1), wid = threadIdx.x / BG_WAVE;
    if (lane == 0) {
        c.dred[wid] = sx;
        c.dred[kWaves + wid] = sy;
    }
    __syncthreads();
    double tx = 0.0, ty = 0.0;
    for (int w = 0; w < kWaves; ++w) {
        tx += c.dred[w];
        ty += c.dred[kWaves + w];
    }
    __syncthreads();
    const double n = W.nb > 0 ? (double)W.nb : 1.0;
    return make_double2(tx / n, ty / n);
}
// Before a launch's first substep.
static __device__ __forceinline__ void start_walk(Ctx& c, Walk& w, const DiffWorld& W) {
    w.skin = kSkin * 2.0f * W.rmax;
    w.drift = make_float2(0.0f, 0.0f);
    w.grid = 0;
    w.tested = 0;
    w.build = true;
    if (threadIdx.x == 0) c.out->n = c.out->pairs[0] = c.out->pairs[1] = 0;
    if (threadIdx.x < 2 * kOutMax) c.out->count[threadIdx.x / kOutMax][threadIdx.x % kOutMax] = 0;
}
};  // Rollout

// With the kernels' own arrays nearly the CU's 160 KB: one workgroup a CU either way (1,024 threads
// at 128 VGPRs fill its registers).
#define BG_DIFF_SHARED                                               \
    using X = Rollout<NT, PER>;                                      \
    constexpr uint32_t kDiffMaxBodies = X::kDiffMaxBodies, kDiffLdsSprings = X::kDiffLdsSprings;       \
    constexpr int kWaves = X::kWaves;                                \
    __shared__ float2 s_xy[kDiffMaxBodies];                          \
    __shared__ float2 s_vel[kDiffMaxBodies];                         \
    __shared__ float s_mass[kDiffMaxBodies], s_rad[kDiffMaxBodies];  \
    __shared__ float4 s_force[kDiffLdsSprings + kLdsRecPad];         \
    __shared__ typename X::JointStage s_joints;                      \
    static_assert(kDiffLdsSprings >= kDiffMaxBodies, "the adjoint vectors and the records share the springs' memory"); \
    typename X::Ctx c{};                                                         \
    c.xy = s_xy;                                                     \
    c.vel = s_vel;                                                   \
    c.mass = s_mass;                                                 \
    c.rad = s_rad;                                                   \
    c.force = s_force;                                               \
    c.joints = &s_joints;                                            \
    c.lam_pp = reinterpret_cast<float2*>(s_force);                   \
    c.lam_am = c.lam_pp + kDiffMaxBodies;

// The forward's.  The scans' and the centroid's scratch is the idle queue's.
#define BG_DIFF_FORWARD                                              \
    BG_DIFF_SHARED                                                   \
    constexpr uint32_t kPairs = X::kPairs, kQueue = kPairs + X::kOutMax * X::kOutPairs;                   \
    __shared__ float s_gmod[kDiffMaxBodies];                         \
    __shared__ float4 s_lists[kDiffMaxBodies + kLdsRecPad];          \
    __shared__ uint32_t s_cnt[X::kDiffCells + 1];                    \
    __shared__ float2 s_res[kQueue];                                 \
    __shared__ uint32_t s_entries[kQueue];                           \
    __shared__ typename X::Outliers s_out;                                       \
    __shared__ LdsGrid s_grid;                                       \
    static_assert(sizeof(uint16_t[X::kListCap / 4][kDiffMaxBodies][4]) <= sizeof(s_lists), "lists, or records"); \
    static_assert(kQueue >= kFitWords * kWaves && kQueue >= 2 * kWaves, "the scratch");                  \
    c.gmod = s_gmod;                                                 \
    c.lists = reinterpret_cast<uint16_t(*)[kDiffMaxBodies][4]>(s_lists); \
    c.cnt = s_cnt;                                                   \
    c.res = s_res;                                                   \
    c.entries = s_entries;                                           \
    c.out = &s_out;                                                  \
    c.grid = &s_grid;                                                \
    c.red = s_entries;                                               \
    c.dred = reinterpret_cast<double*>(s_res);                       \
    typename X::Walk w;

template <uint32_t NT, uint32_t PER>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_diff_forward(DiffArgs a, uint32_t n_steps, uint32_t ck_every) {
    BG_DIFF_FORWARD
    const DiffWorld W = a.worlds[blockIdx.x];
    typename X::Own o;
    X::load_own(c, o, a, W, a.ck_p, a.ck_q, a.ck_v);
    X::start_walk(c, w, W);
    __syncthreads();
    for (uint32_t step = 0; step < n_steps; ++step) {
        if (step > 0 && step % ck_every == 0) {
            const size_t base = (size_t)(step / ck_every) * a.nb_total + W.b0;
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j)
                if (threadIdx.x + j * NT < W.nb) {
                    a.ck_p[base + threadIdx.x + j * NT] = o.p[j];
                    a.ck_q[base + threadIdx.x + j * NT] = o.q[j];
                    a.ck_v[base + threadIdx.x + j * NT] = c.vel[threadIdx.x + j * NT];
                }
        }
        for (uint32_t sub = 0; sub < a.substeps; ++sub) {
            const uint32_t n = step * a.substeps + sub;
            X::template substep_forward<false>(c, o, w, a, W, n, n, 0u);
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j)
        if (threadIdx.x + j * NT < W.nb) a.final_p[W.b0 + threadIdx.x + j * NT] = o.p[j];
    const double2 cen = X::block_centroid(c, o, W);
    if (threadIdx.x == 0) {
        const double dx = cen.x - (double)W.tx, dy = cen.y - (double)W.ty;
        a.loss[blockIdx.x] = (float)(dx * dx + dy * dy);
    }
}

// Recomputes segments first_seg + blockIdx.y from their checkpoints, recording their tapes
// one after another (seg_sub substeps each).
template <uint32_t NT, uint32_t PER>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_diff_recompute(DiffArgs a, uint32_t first_seg, uint32_t ck_every,
                                                                 uint32_t n_steps) {
    BG_DIFF_FORWARD
    const DiffWorld W = a.worlds[blockIdx.x];
    const uint32_t seg = first_seg + blockIdx.y, first_step = seg * ck_every;
    const uint32_t nsub = min(n_steps - first_step, ck_every) * a.substeps;
    const uint32_t tape0 = blockIdx.y * ck_every * a.substeps;
    const size_t ck = (size_t)seg * a.nb_total;
    typename X::Own o;
    X::load_own(c, o, a, W, a.ck_p + ck, a.ck_q + ck, a.ck_v + ck);
    X::start_walk(c, w, W);
    __syncthreads();
    for (uint32_t k = 0; k < nsub; ++k)
        X::template substep_forward<true>(c, o, w, a, W, first_step * a.substeps + k, k, tape0 + k);
}

// Adjoint of one segment, its tape at slots tape0 ...
template <uint32_t NT, uint32_t PER>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_diff_reverse(DiffArgs a, uint32_t seg, uint32_t tape0,
                                                               uint32_t first_sub, uint32_t nsub, uint32_t last) {
    BG_DIFF_SHARED
    __shared__ float4 s_rec[kDiffMaxBodies];
    __shared__ float2 s_spring_k[kDiffLdsSprings], s_spring_v[PER == 1 ? kDiffLdsSprings : 1];
    __shared__ float2 s_axes[X::kDiffLdsSolves];
    __shared__ double s_dred[2 * kWaves];
    c.rec = s_rec;
    c.spring_k = s_spring_k;
    c.spring_v = PER == 1 ? s_spring_v : s_xy;
    static_assert(PER == 1 || kDiffMaxBodies >= kDiffLdsSprings, "spring adjoints in the positions' memory");
    c.axes = s_axes;
    c.dred = s_dred;
    const DiffWorld W = a.worlds[blockIdx.x];
    typename X::Own o;
    // (only the last segment reads positions: the final ones, for the centroid)
    X::load_own(c, o, a, W, a.final_p, a.final_p, a.final_p);
    __syncthreads();
    float2 lp[PER], lq[PER], lv[PER], gv[PER];
    const bool centroid = last && !a.dl_dfinal;
    float2 g0 = make_float2(0.0f, 0.0f);
    if (centroid) {  // d |centroid - target|^2 / d p_i = 2 (centroid - target) / n
        const double2 cen = X::block_centroid(c, o, W);
        g0.x = (float)(2.0 * (cen.x - (double)W.tx) / (double)(W.nb > 0 ? W.nb : 1));
        g0.y = (float)(2.0 * (cen.y - (double)W.ty) / (double)(W.nb > 0 ? W.nb : 1));
    }
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        const uint32_t li = threadIdx.x + j * NT, gi = W.b0 + li;
        const bool live = li < W.nb;
        lp[j] = centroid ? g0 : (live ? (last ? a.dl_dfinal[gi] : a.lam_p[gi]) : make_float2(0.0f, 0.0f));
        lq[j] = (live && !last) ? a.lam_q[gi] : make_float2(0.0f, 0.0f);
        lv[j] = (live && !last) ? a.lam_v[gi] : make_float2(0.0f, 0.0f);  // the loss does not read the final velocities
        gv[j] = make_float2(0.0f, 0.0f);
    }
    const bool own_gk = X::lds_springs(W) && threadIdx.x < W.ns;
    float gk = own_gk ? a.grad_k[W.s0 + threadIdx.x] : 0.0f;
    typename X::Tape t;
    if (nsub > 0) X::load_tape(t, a, W, tape0 + nsub - 1);
    for (uint32_t k = nsub; k-- > 0;)
        X::substep_reverse(c, o, a, W, first_sub + k, tape0 + k, k > 0, t, lp, lq, lv, gv, gk);
    if (own_gk) a.grad_k[W.s0 + threadIdx.x] = gk;
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        const uint32_t li = threadIdx.x + j * NT, gi = W.b0 + li;
        if (li >= W.nb) continue;
        a.lam_p[gi] = lp[j];
        a.lam_q[gi] = lq[j];
        a.lam_v[gi] = lv[j];
        if (seg == 0) a.grad_vreq[gi] = gv[j];
    }
}

}  // namespace

#define BG_DIFF_LAUNCH(KERNEL, GRID, ...)                                                                     \
    do {                                                                                                      \
        switch (a.threads) {                                                                                  \
            case 256: KERNEL<256, 1><<<GRID, 256, 0, s>>>(__VA_ARGS__); break;                                \
            case 512: KERNEL<512, 1><<<GRID, 512, 0, s>>>(__VA_ARGS__); break;                                \
            case 1024: KERNEL<1024, 1><<<GRID, 1024, 0, s>>>(__VA_ARGS__); break;                             \
            default: KERNEL<kDiffThreads, kDiffPer><<<GRID, kDiffThreads, 0, s>>>(__VA_ARGS__); break;        \
        }                                                                                                     \
    } while (0)

hipError_t launch_diff_forward(const DiffArgs& a, uint32_t n_steps, uint32_t ck_every, hipStream_t s) {
    if (a.n_worlds == 0) return hipSuccess;
    BG_DIFF_LAUNCH(k_diff_forward, a.n_worlds, a, n_steps, ck_every);
    return hipGetLastError();
}

hipError_t launch_diff_recompute(const DiffArgs& a, uint32_t first_seg, uint32_t n_seg, uint32_t ck_every,
                                 uint32_t n_steps, hipStream_t s) {
    if (a.n_worlds == 0) return hipSuccess;
    BG_DIFF_LAUNCH(k_diff_recompute, dim3(a.n_worlds, n_seg), a, first_seg, ck_every, n_steps);
    return hipGetLastError();
}

hipError_t launch_diff_reverse(const DiffArgs& a, uint32_t seg, uint32_t tape_seg, uint32_t ck_every, uint32_t n_steps,
                               hipStream_t s) {
    if (a.n_worlds == 0) return hipSuccess;
    const uint32_t first = seg * ck_every, steps = std::min(n_steps - first, ck_every);
    BG_DIFF_LAUNCH(k_diff_reverse, a.n_worlds, a, seg, tape_seg * ck_every * a.substeps, first * a.substeps,
                   steps * a.substeps, first + steps == n_steps ? 1u : 0u);
    return hipGetLastError();
}

}  // namespace bg
