// small_kernels.hip -- worlds of at most kSmallBodies single centred spheres
// (a plain world, or every world of a batch): one workgroup advances a world
// through every substep of a launch, a body a thread, its state in registers
// and the snapshot in LDS.
//
// The substep is the fused sphere path's (physics.rs:401-421 for one collider
// per body, no springs or joints): gravity, contacts against the substep's
// snapshot summed in ascending partner id (physics.rs:241-317; push-outs by the
// pair rule, flagged), Verlet with the world's own old_dt (Q1,
// physics.rs:326-358), collider transform (physics.rs:360-366), circle
// constraints (physics.rs:377-395).  The same f32 operations in the same order
// as the grid path's kernels, so a world evolves bit-identically on either.
//
// Partner lists.  A world this small is bound by the chain of dependent LDS
// reads and barriers of a substep, not by arithmetic or memory, so the cell
// grid (fit, count, scan, scatter, walk: nine barriers) is built only when a body
// has left its skin, and collects for each body the partners it could touch
// until then: bodies a and b with skins s_a and s_b can be in contact only if
// their positions at the build were within r_a + r_b + s_a + s_b, after the
// world's common motion (the mean displacement of its dynamic bodies a substep,
// which cancels within a pair).  A body's skin is what it travels in
// kSkinSubsteps substeps, at least kSkinRest and at most kSkinMax diameters, so a
// few fast bodies lengthen their own lists and their neighbours', not everyone's.
// Which candidates are tested never changes a result.
//
// A steady substep has three phases with a barrier after each: mark (list
// entries within reach go into a queue), correct (a queued pair a thread), sum
// and integrate.  The lists are sorted once, at the build, so a body's entries
// are in ascending partner id and the sum is one pass; the snapshot is 8 bytes a
// body apart from radius and mass, because gathers of 16 are bound by LDS banks.
//
// Measured (cycles of one wave): a steady substep 2,800 at 100 free bodies,
// 4,900 at 500, 11,700 at 2,000, 7,500 at the 364 of a settled pile (12,000 with
// unsorted lists summed by selection); a build 13,000, 18,000, 49,000.  One step of
// 8 substeps: 364 bodies 127 us on the grid path (14 launches) and 47 here;
// 128 worlds of 64 to 512 106 and 31.
#include "common.hpp"
#include "device_state.hpp"
#include "lds_grid.hpp"
#include "step_common.hpp"

namespace bg {

namespace {

constexpr uint32_t kListCap = 16;      // partners of a list; a body with more is tested against every body
constexpr uint32_t kListGroups = kListCap / 4;
constexpr float kSkinSubsteps = 8.0f;  // substeps a list is meant to last
// Least and largest skin, in diameters of the largest body.  At 1,024 worlds of 64 to 1,024 a step
// takes 112 us; with 0.05 and 0.25 146, 0.1 and 0.1 182, 0.1 and 0.5 115, 12 substeps 110 -- but
// 1,288 bodies falling on a pile 225 then, instead of 142 (0.05 and 0.25: 211).
constexpr float kSkinRest = 0.1f;
constexpr float kSkinMax = 1.0f;
constexpr uint32_t kListTries = 4;     // builds with skins halved while lists overflow
// A list that overflows for one body in so many threads is left so: lists with smaller skins last
// shorter, for everyone.  A step of 300, 1,000 and 2,000 bodies of ragged radii under one of 24
// times their size takes 426, 956 and 2,137 us (929, 1,591, 3,546 with none left); of 2,000 pressed into a
// circle 1,417 (1,406, and 1,456 with one in 64).
constexpr uint32_t kListsOver = 256;
constexpr uint32_t kFast = 0x10000u;   // record flag: more than the least skin
constexpr float kMaxDrift = 16.0f;     // common motion a list is kept for (rounding of x - x0 - drift)

// The queue of pairs lives from the mark phase to the sums, the grid only during a build.
template <uint32_t NT, uint32_t PER>
union SmallScratch {
    static constexpr uint32_t kBodies = NT * PER, kCap = 4 * NT, kCells = PER == 1 ? 6 * NT : 3 * NT;
    struct {
        float2 res[kCap];
        uint32_t entries[kCap];
    } q;
    struct {
        float4 rec[kBodies + kLdsRecPad];  // (x, y, radius + skin, bits(local index | kFast)) in cell order
        uint32_t start[kCells + 1];
        uint32_t red[kFitWords * (NT / BG_WAVE)];
    } b;
};

// A thread's bodies, those of slots t + j * NT of the world.  With two, the phases loop over them
// at run time and pick the state by selects: unrolled, two contact passes in flight spill.
template <uint32_t PER>
struct Own {
    float2 p[PER], q[PER], rw[PER], x0[PER];  // x0: snapshot of the last build, NaN if it was not finite
    float gm[PER], skin[PER];
    uint32_t id[PER];  // local index | body flags << 16
};
__device__ __forceinline__ float lane_f32(float v, int lane) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane));
}

// Sorts the first n (at most N) partners of body li's list and fills up to N with li, by
// Batcher's odd-even merge network (every index a constant, so the list is in registers).
template <uint32_t N, uint32_t B>
__device__ __forceinline__ void sort_list(uint16_t (&lists)[kListGroups][B][4], uint32_t li, uint32_t n, bool live) {
    uint32_t v[N];
#pragma unroll
    for (uint32_t c = 0; c < N / 4; ++c) {
        const uint2 l = *(const uint2*)lists[c][li];
        v[4 * c] = l.x & 0xFFFFu;
        v[4 * c + 1] = l.x >> 16;
        v[4 * c + 2] = l.y & 0xFFFFu;
        v[4 * c + 3] = l.y >> 16;
    }
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) v[i] = i < n ? v[i] : 0xFFFFu;
#pragma unroll
    for (uint32_t p = 1; p < N; p *= 2)
#pragma unroll
        for (uint32_t q = p; q >= 1; q /= 2)
#pragma unroll
            for (uint32_t a = q % p; a + q < N; a += 2 * q)
#pragma unroll
                for (uint32_t i = a; i < a + q && i + q < N; ++i)
                    if (i / (2 * p) == (i + q) / (2 * p)) {
                        const uint32_t lo = min(v[i], v[i + q]), hi = max(v[i], v[i + q]);
                        v[i] = lo;
                        v[i + q] = hi;
                    }
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) v[i] = i < n ? v[i] : li;
    if (!live) return;
#pragma unroll
    for (uint32_t c = 0; c < N / 4; ++c)
        *(uint2*)lists[c][li] = make_uint2(v[4 * c] | v[4 * c + 1] << 16, v[4 * c + 2] | v[4 * c + 3] << 16);
}

template <uint32_t NT, uint32_t PER, bool EVENTS>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_small_step(SmallArgs k, const uint32_t* __restrict__ order) {
    using Scratch = SmallScratch<NT, PER>;
    constexpr uint32_t B = NT * PER;
    static_assert(PER <= 2 && B <= 0x10000u, "picks; 16-bit indices");
    constexpr bool kVelLds = EVENTS && PER == 1;               // (LDS is full with two bodies a thread)
    __shared__ float2 xy[B], rm[B];                            // snapshot; (radius, mass): by local index
    __shared__ alignas(8) uint16_t lists[kListGroups][B][4];   // partners by local index
    __shared__ uint32_t n_list[B];
    __shared__ float2 vs[kVelLds ? B : 1];                     // velocities before the contact pass
    __shared__ Scratch sc;
    __shared__ LdsGrid s_grid;
    // by substep parity: a body left its skin; queued pairs; a body's contacts are worked out directly
    __shared__ uint32_t s_left[2], s_count[2], s_direct[2];
    __shared__ uint32_t s_rmax, s_rmin, s_fast;

    const uint32_t t = threadIdx.x, lane = t & (BG_WAVE - 1);
    const uint32_t w = order[blockIdx.x];
    const uint32_t b0 = k.wstart[w], nb = min(k.wstart[w + 1] - b0, B);
    const uint32_t per = PER == 1 || nb <= NT ? 1u : PER;

    Own<PER> o;
    float wold = 0.0f;
    uint32_t most = 0, least = 0xFFFFFFFFu;  // f2ord of the radii
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        o.p[j] = o.q[j] = o.rw[j] = o.x0[j] = make_float2(0.0f, 0.0f);
        o.gm[j] = o.skin[j] = 0.0f;
        o.id[j] = 0u;
        if (t + j * NT >= nb) continue;
        const uint32_t g = b0 + t + j * NT;
        const float4 s = k.s.snap[g], pp = k.s.pp[g];
        const float2 mg = k.s.mg[g];
        const uint32_t fl = k.s.bflags[g];
        // slots may have been permuted by the grid path
        const uint32_t word = __float_as_uint(s.w) & (k.snap_flags ? kSnapIdMask : ~kSnapOutlier);
        const uint32_t li = min(word - b0, B - 1u);
        o.p[j] = make_float2(pp.x, pp.y);
        o.q[j] = make_float2(pp.z, pp.w);
        o.rw[j] = k.s.rw[g];
        o.gm[j] = mg.y;
        o.id[j] = li | fl << 16;
        xy[li] = make_float2(s.x, s.y);
        rm[li] = make_float2(s.z, mg.x);
        most = max(most, f2ord(s.z));
        least = min(least, f2ord(s.z));
        if (fl & BF_FIRST_DYN) wold = k.wold_dt[w];
        if (EVENTS) {
            if (kVelLds)
                vs[li] = k.s.vel[g];
            else
                k.vel_scratch[b0 + li] = k.s.vel[g];
        }
    }
    if (t == 0) {
        s_left[0] = s_left[1] = s_count[0] = s_count[1] = s_direct[0] = s_direct[1] = 0u;
        s_rmax = 0u;
        s_rmin = 0xFFFFFFFFu;
    }
    __syncthreads();
    most = wave_prefix(most, 0u, MaxU32());
    least = wave_prefix(least, 0xFFFFFFFFu, MinU32());
    if (lane == BG_WAVE - 1) {
        atomicMax(&s_rmax, most);
        atomicMin(&s_rmin, least);
    }
    __syncthreads();
    const float rmax = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(ord2f(s_rmax))));
    const bool alike = s_rmax == s_rmin;  // one radius: the mark phase needs no partner's
    float span = kSkinSubsteps, rest = kSkinRest * 2.0f * rmax;
    uint32_t age = 0;  // substeps since the build
    float2 drift = make_float2(0.0f, 0.0f);
    bool build = true;
    uint32_t count = 0, pushes = 0, flags = 0;

    auto tally = [&](uint32_t own, uint32_t other, const LdsContact& c, uint32_t sub) {
        const bool is_a = own > other;
        if (is_a) ++count;
        if (c.pushed) {
            ++pushes;
            flags |= INFO_PUSH_OUT;
        }
        if (c.nan) flags |= ERR_NAN_NORMAL;
        if (EVENTS && is_a) {
            const unsigned long long e = atomicAdd(&k.accum->event_count, 1ull);
            if (e < k.event_cap) {
                DevEvent ev;
                ev.sub = k.sub_global + sub;
                ev.a = b0 + own;
                ev.b = b0 + other;
                ev.pad = 0;
                ev.va = kVelLds ? vs[kVelLds ? own : 0] : k.vel_scratch[b0 + own];
                ev.vb = kVelLds ? vs[kVelLds ? other : 0] : k.vel_scratch[b0 + other];
                k.events[e] = ev;
            }
        }
    };
    // the contact of two bodies, from the side of `own`
    auto contact = [&](uint32_t own, uint32_t other) {
        const float2 a = xy[own], b = xy[other], ra = rm[own], rb = rm[other];
        return lds_correction(make_float4(a.x, a.y, ra.x, 0.0f), make_float4(b.x, b.y, rb.x, 0.0f), ra.y, rb.y,
                              own > other, false);
    };
    // whether they can be one
    auto near = [&](uint32_t own, uint32_t other) -> uint32_t {
        const float2 a = xy[own], b = xy[other];
        const float dx = a.x - b.x, dy = a.y - b.y, r = rm[own].x, rs = r + (alike ? r : rm[other].x);
        return dx * dx + dy * dy > (rs * rs) * 1.00000095367431640625f ? 0u : 1u;
    };
    auto append = [&](uint32_t to, uint32_t partner) {
        const uint32_t at = atomicAdd(&n_list[to], 1u);
        if (at < kListCap) lists[at >> 2][to][at & 3u] = (uint16_t)partner;
    };

    for (uint32_t sub = 0; sub < k.nsub; ++sub) {
        uint32_t t = threadIdx.x;
        asm volatile("" : "+v"(t));  // (or what is derived from it is kept from phase to phase, and spills)
        const bool fresh = k.fresh && sub == 0;
        const uint32_t par = sub & 1u;
        LdsPairs pr[PER];
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) pr[j] = LdsPairs{0, 0, false};
        if (k.collisions && build) {
            // a body's displacement a substep
            auto moving = [&](uint32_t j, uint32_t fl) {
                const float2 p = pick(o.p, j), q = pick(o.q, j);
                if (sub == 0 && (fl & BF_HAS_VREQ)) {
                    const float2 v = k.s.vreq[b0 + t + j * NT];
                    return make_float2(v.x * k.h, v.y * k.h);
                }
                return make_float2(p.x - q.x, p.y - q.y);
            };
            LdsFit fit;
            fit.init();
#pragma unroll 1
            for (uint32_t j = 0; j < per; ++j) {
                if (t + j * NT >= nb) continue;
                const uint32_t id = pick(o.id, j), fl = id >> 16;
                const float2 own = xy[id & 0xFFFFu];
                fit.point(own.x, own.y);
                const float2 d = moving(j, fl);
                if (!(fl & BF_STATIC)) fit.extra(d.x, d.y);
                const bool fin = finitef(own.x) && finitef(own.y);
                put(o.x0, j, make_float2(fin ? own.x : __uint_as_float(0x7FC00000u), own.y));
            }
            lds_fit<NT>(fit, 2.004f * (rmax + rest), Scratch::kCells, sc.b.red, &s_grid);
            const LdsGrid gr = lds_grid_uniform(s_grid);
            drift = make_float2(gr.ex, gr.ey);
            age = 0;
            for (uint32_t i = t; i <= gr.ncells; i += NT) sc.b.start[i] = 0u;
            __syncthreads();
            const float margin = 1e-4f * (2.0f * rmax + 2.0f * rest) + 1e-5f;
            uint32_t at[PER];  // cell, then slot in cell order
            uint32_t rank[PER];
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                at[j] = 0u;
                rank[j] = kNoPair;
                if (t + j * NT >= nb || !(o.x0[j].x == o.x0[j].x)) continue;
                at[j] = lds_cell(gr, o.x0[j].x, o.x0[j].y);
                rank[j] = atomicAdd(&sc.b.start[at[j]], 1u);
            }
            __syncthreads();
            lds_scan<NT, (Scratch::kCells + NT) / NT>(sc.b.start, gr.ncells + 1u, sc.b.red);
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j)
                at[j] = rank[j] != kNoPair ? sc.b.start[at[j]] + rank[j] : kNoPair;
            for (uint32_t tries = 1;; ++tries) {
                if (t == 0) s_fast = 0u;
#pragma unroll 1
                for (uint32_t j = 0; j < per; ++j) {
                    if (t + j * NT >= nb) continue;
                    const uint32_t id = pick(o.id, j), li = id & 0xFFFFu;
                    const float2 d = moving(j, id >> 16);
                    float skin = 1.125f * span * vlen(d.x - drift.x, d.y - drift.y);
                    skin = fminf(fmaxf(rest, skin), kSkinMax * 2.0f * rmax);
                    if (!(skin >= rest)) skin = rest;
                    put(o.skin, j, skin);
                    const uint32_t a = pick(at, j);
                    if (a != kNoPair) {
                        const float2 own = xy[li];
                        sc.b.rec[a] = make_float4(own.x, own.y, rm[li].x + skin,
                                                  __uint_as_float(li | (skin > rest ? kFast : 0u)));
                    }
                }
                __syncthreads();
                // Bodies of the least skin find each other, each its own list.
#pragma unroll 1
                for (uint32_t j = 0; j < per; ++j) {
                    if (t + j * NT >= nb) continue;
                    const uint32_t a = pick(at, j), li = pick(o.id, j) & 0xFFFFu;
                    const float skin = pick(o.skin, j);
                    if (a == kNoPair || skin > rest) {
                        n_list[li] = 0u;
                        if (a != kNoPair) s_fast = 1u;
                        continue;
                    }
                    const float2 own = xy[li];
                    const float reach = rm[li].x + rest + margin, Q = reach + rmax + rest;
                    auto near = [&](uint32_t u, const float4& b) {
                        const float dx = own.x - b.x, dy = own.y - b.y, rs = reach + b.z;
                        return !((u == a) | (dx * dx + dy * dy > rs * rs) | ((__float_as_uint(b.w) & kFast) != 0u));
                    };
                    uint32_t n = 0;
                    auto take = [&](uint32_t u) {
                        if (n < kListCap) lists[n >> 2][li][n & 3u] = (uint16_t)__float_as_uint(sc.b.rec[u].w);
                        ++n;
                    };
                    const LdsRows l = lds_rows(gr, sc.b.start, true, own, Q);
                    if (l.flat) {
                        for (uint64_t m = lds_near(l, sc.b.rec, near); m != 0; m &= m - 1)
                            take(l.slot((uint32_t)__builtin_ctzll(m)));
                    } else {
                        const LdsRect c = lds_rect(gr, own.x, own.y, Q);
                        for (int32_t cy = c.cy0; cy <= c.cy1; ++cy) {
                            const uint32_t row = (uint32_t)cy * (uint32_t)gr.nx;
                            const uint32_t u1 = sc.b.start[row + (uint32_t)c.cx1 + 1u];
                            for (uint32_t u = sc.b.start[row + (uint32_t)c.cx0]; u < u1; ++u)
                                if (near(u, sc.b.rec[u])) take(u);
                        }
                    }
                    n_list[li] = n;
                }
                __syncthreads();
                if (s_fast) {
                    // A fast body finds its slow partners, and the fast ones of smaller reach (then
                    // index): its walk covers those.  Such a pair goes to both lists.
#pragma unroll 1
                    for (uint32_t j = 0; j < per; ++j) {
                        const float skin = pick(o.skin, j);
                        const uint32_t a = pick(at, j);
                        if (t + j * NT >= nb || a == kNoPair || !(skin > rest)) continue;
                        const uint32_t li = pick(o.id, j) & 0xFFFFu;
                        const float2 own = xy[li];
                        const float z = rm[li].x + skin;
                        const float reach = z + (1e-4f * (z + fmaxf(z, rmax + rest)) + 1e-5f);
                        const LdsRect c = lds_rect(gr, own.x, own.y, reach + fmaxf(z, rmax + rest));
                        for (int32_t cy = c.cy0; cy <= c.cy1; ++cy) {
                            const uint32_t row = (uint32_t)cy * (uint32_t)gr.nx;
                            const uint32_t u1 = sc.b.start[row + (uint32_t)c.cx1 + 1u];
                            for (uint32_t u = sc.b.start[row + (uint32_t)c.cx0]; u < u1; u += 4) {
                                float4 b[4];
#pragma unroll
                                for (uint32_t i = 0; i < 4; ++i) b[i] = sc.b.rec[u + i];
#pragma unroll
                                for (uint32_t i = 0; i < 4; ++i) {
                                    const float dx = own.x - b[i].x, dy = own.y - b[i].y, rs = reach + b[i].z;
                                    if ((u + i >= u1) | (u + i == a) | (dx * dx + dy * dy > rs * rs)) continue;
                                    const uint32_t lj = __float_as_uint(b[i].w) & 0xFFFFu;
                                    if ((__float_as_uint(b[i].w) & kFast) &&
                                        (b[i].z > z || (b[i].z == z && lj > li)))
                                        continue;
                                    append(li, lj);
                                    append(lj, li);
                                }
                            }
                        }
                    }
                    __syncthreads();
                }
                bool over = false;
#pragma unroll
                for (uint32_t j = 0; j < PER; ++j)
                    over |= t + j * NT < nb && n_list[o.id[j] & 0xFFFFu] > kListCap;
                if (__syncthreads_count(over) <= (int)(NT / kListsOver) || tries == kListTries) break;
                span *= 0.5f;
                rest *= 0.5f;
            }
            // ascending, the rest of the last group filled with the body itself
#pragma unroll 1
            for (uint32_t j = 0; j < per; ++j) {
                const bool live = t + j * NT < nb;
                const uint32_t li = pick(o.id, j) & 0xFFFFu, n = live ? min(n_list[li], kListCap) : 0u;
                if (__any(n > 8u))
                    sort_list<16>(lists, li, n, live);
                else
                    sort_list<8>(lists, li, n, live);
            }
        }
        if (k.collisions) {
            // mark
#pragma unroll 1
            for (uint32_t j = 0; j < per; ++j) {
                uint32_t marked = 0, n = 0, li = 0;
                bool all = false;
                if (t + j * NT < nb) {
                    li = pick(o.id, j) & 0xFFFFu;
                    const float2 own = xy[li];
                    n = n_list[li];
                    const bool fin = finitef(own.x) && finitef(own.y);
                    all = fin && n > kListCap;
                    if (!fin || all) n = 0;
                    for (uint32_t f = 0; f < n; f += 4) {
                        const uint2 l = *(const uint2*)lists[f >> 2][li];
                        marked |= (near(li, l.x & 0xFFFFu) | near(li, l.x >> 16) << 1 | near(li, l.y & 0xFFFFu) << 2 |
                                   near(li, l.y >> 16) << 3) << f;
                    }
                    marked &= (1u << n) - 1u;
                    static_assert(kListCap < 32, "the mask");
                }
                LdsPairs r = lds_queue<Scratch::kCap>(marked, li, sc.q.entries, &s_count[par],
                                                      [](uint32_t i) { return i; });
                r.direct |= all;
                if (__any(r.direct) && lane == 0) s_direct[par] = 1u;
                if (PER == 1 || j == 0)
                    pr[0] = r;
                else
                    pr[PER - 1] = r;
            }
            __syncthreads();
            // correct
            for (uint32_t e = t; e < min(s_count[par], Scratch::kCap); e += NT) {
                const uint32_t pair = sc.q.entries[e];
                if (pair == kNoPair) continue;
                const uint32_t own = pair >> 16, i = pair & 0xFFFFu;
                const uint32_t other = lists[i >> 2][own][i & 3u];
                const LdsContact c = contact(own, other);
                if (!c.hit) sc.q.entries[e] = kNoPair;
                sc.q.res[e] = c.c;
                if (c.hit) tally(own, other, c, sub);
            }
            __syncthreads();
            if (s_direct[par]) {
                // No room in the queue: the body's thread works its contacts out itself.  A list that
                // overflowed: the body's wave tests it against everyone, a partner a lane, one such body
                // after the other.  Both in ascending partner index.
#pragma unroll 1
                for (uint32_t j = 0; j < per; ++j) {
                    const bool direct = t + j * NT < nb && (PER == 1 || j == 0 ? pr[0].direct : pr[PER - 1].direct);
                    const uint32_t li = pick(o.id, j) & 0xFFFFu, n = direct ? n_list[li] : 0u;
                    float2 p = pick(o.p, j);
                    uint32_t within = 0;
                    for (uint32_t i = 0; i < (n > kListCap ? 0u : n); ++i) within |= near(li, lists[i >> 2][li][i & 3u]) << i;
                    for (; within != 0; within &= within - 1) {
                        const uint32_t i = (uint32_t)__builtin_ctz(within), lj = lists[i >> 2][li][i & 3u];
                        const LdsContact c = contact(li, lj);
                        if (!c.hit) continue;
                        tally(li, lj, c, sub);
                        p.x = p.x + c.c.x;
                        p.y = p.y + c.c.y;
                    }
                    for (uint64_t left = __ballot(n > kListCap); left != 0; left &= left - 1) {
                        const int of = __builtin_ctzll(left);
                        const uint32_t own = (uint32_t)__builtin_amdgcn_readlane((int)li, of);
                        float2 q = make_float2(lane_f32(p.x, of), lane_f32(p.y, of));
                        for (uint32_t first = 0; first < nb; first += BG_WAVE) {
                            const uint32_t lj = first + lane;
                            LdsContact c = {make_float2(0.0f, 0.0f), false, false, false};
                            if (lj < nb && lj != own) c = contact(own, lj);
                            if (c.hit) tally(own, lj, c, sub);
                            for (uint64_t hits = __ballot(c.hit); hits != 0; hits &= hits - 1) {
                                const int h = __builtin_ctzll(hits);
                                q.x = q.x + lane_f32(c.c.x, h);
                                q.y = q.y + lane_f32(c.c.y, h);
                            }
                        }
                        if ((int)lane == of) p = q;
                    }
                    if (direct) put(o.p, j, p);
                }
                __syncthreads();  // before anyone publishes
            }
        }
        // sum, update_objects (physics.rs:326-358), collider transform, constraints
        bool left = false;
        ++age;
#pragma unroll 1
        for (uint32_t j = 0; j < per; ++j) {
            if (t + j * NT >= nb) continue;
            const uint32_t g = b0 + t + j * NT;
            const uint32_t id = pick(o.id, j), li = id & 0xFFFFu, fl = id >> 16;
            BodyState st;
            st.p = pick(o.p, j);
            st.po = pick(o.q, j);
            // (lists are in ascending order, so are a body's entries)
            const uint32_t first = PER == 1 || j == 0 ? pr[0].first : pr[PER - 1].first;
            const uint32_t end = first + (PER == 1 || j == 0 ? pr[0].n : pr[PER - 1].n);
#pragma unroll 4
            for (uint32_t e = first; e < end; ++e) {
                const float2 c = sc.q.res[e];
                const bool hit = sc.q.entries[e] != kNoPair;
                st.p.x = hit ? st.p.x + c.x : st.p.x;
                st.p.y = hit ? st.p.y + c.y : st.p.y;
            }
            const float2 rw = pick(o.rw, j);
            st.rot = rw.x;
            st.omega = rw.y;
            if (fl & BF_STATIC) {
                st.po = st.p;
                st.vel = make_float2(0.0f, 0.0f);
            } else {
                float2 acc = fresh ? k.s.acc[g] : make_float2(0.0f, 0.0f);
                const float gm = pick(o.gm, j);
                acc.x = acc.x + k.gx * gm;
                acc.y = acc.y + k.gy * gm;
                const bool vr = (fl & BF_HAS_VREQ) != 0u;
                const float2 vreq = vr ? k.s.vreq[g] : make_float2(0.0f, 0.0f);
                const float tq = fresh ? k.s.torque[g] : 0.0f;
                const float toi = (fresh || !(fl & BF_INERTIA_POS)) ? tq / k.s.inertia[g] : 0.0f;
                float ratio = k.ratio_rest;
                if (fl & BF_FIRST_DYN) {  // Q1: this world's old_dt
                    ratio = k.h / wold;
                    wold = k.h;
                }
                verlet_dynamic(st, acc, toi, vr, vreq, k.h, ratio);
                if (vr) put(o.id, j, id & ~(BF_HAS_VREQ << 16));
            }
            const float2 x = body_xform_zero_off(st.rot, st.p);
            apply_constraints(st.p, k.con_pos, k.con_r, k.nk);
            put(o.p, j, st.p);
            put(o.q, j, st.po);
            put(o.rw, j, make_float2(st.rot, st.omega));
            xy[li] = x;
            if (kVelLds) vs[kVelLds ? li : 0] = st.vel;
            if (EVENTS && !kVelLds) k.vel_scratch[b0 + li] = st.vel;
            if (sub + 1 == k.nsub) k.s.vel[g] = st.vel;
            const float2 x0 = pick(o.x0, j);
            const float skin = pick(o.skin, j);
            const float dx = (x.x - x0.x) - (float)age * drift.x, dy = (x.y - x0.y) - (float)age * drift.y;
            left |= finitef(x.x) && finitef(x.y) && !(dx * dx + dy * dy <= skin * skin);
        }
        left |= !((float)age * (fabsf(drift.x) + fabsf(drift.y)) <= kMaxDrift);
        if (__any(left) && lane == 0) s_left[par] = 1u;
        if (t == 0) s_left[par ^ 1u] = s_count[par ^ 1u] = s_direct[par ^ 1u] = 0u;
        __syncthreads();
        build = __builtin_amdgcn_readfirstlane((int)s_left[par]) != 0;
    }
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        if (t + j * NT >= nb || k.nsub == 0) continue;
        const uint32_t g = b0 + t + j * NT, li = o.id[j] & 0xFFFFu;
        uint32_t fl = o.id[j] >> 16;
        const float2 rw = o.rw[j];
        const bool still = (fl & BF_STATIC) != 0u ||
                           (__float_as_uint(rw.y) == 0u && __float_as_uint(rw.x) != 0x80000000u && finitef(rw.x) &&
                            (fl & BF_INERTIA_POS) != 0u);
        fl = still ? (fl | BF_ROT_STILL) : (fl & ~BF_ROT_STILL);
        const uint32_t word = (b0 + li) | (k.snap_flags ? (fl & kSnapFlagMask) << kSnapFlagShift : 0u);
        k.s.snap[g] = make_float4(xy[li].x, xy[li].y, rm[li].x, __uint_as_float(word));
        k.s.pp[g] = make_float4(o.p[j].x, o.p[j].y, o.q[j].x, o.q[j].y);
        k.s.rw[g] = rw;
        k.s.bflags[g] = fl;
        if (k.fresh && !(fl & BF_STATIC)) k.s.torque[g] = 0.0f;
        if (fl & BF_FIRST_DYN) k.wold_dt[w] = wold;
    }
    // counters: contacts into the slot of the world's first body, summed on the host
    if (flags) atomicOr(&k.accum->error_flags, flags);
    const uint32_t c_sum = wave_sum_u32(count), p_sum = wave_sum_u32(pushes);
    if (lane == 0) {
        if (c_sum) atomicAdd(&k.block_contacts[b0 / 64u], (unsigned long long)c_sum);
        if (p_sum) atomicAdd(&k.accum->push_outs, p_sum);
    }
}

template <uint32_t C>
void launch_class(const SmallArgs& k, hipStream_t s) {
    constexpr uint32_t NT = kSmallClassThreads[C], PER = kSmallClassBodies[C] / NT;
    const uint32_t first = k.class_start[C], n = k.class_start[C + 1] - first;
    if (n == 0) return;
    if (k.events)
        k_small_step<NT, PER, true><<<n, NT, 0, s>>>(k, k.order + first);
    else
        k_small_step<NT, PER, false><<<n, NT, 0, s>>>(k, k.order + first);
}

}  // namespace

hipError_t launch_small_step(const SmallArgs& k, hipStream_t s) {
    static_assert(kSmallClasses == 4, "one launch per class");
    launch_class<0>(k, s);
    launch_class<1>(k, s);
    launch_class<2>(k, s);
    launch_class<3>(k, s);
    return hipGetLastError();
}

}  // namespace bg
