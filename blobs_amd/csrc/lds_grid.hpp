// lds_grid.hpp -- contacts of one world inside one workgroup: its bodies'
// snapshot filed by cell in LDS, from which partner lists are filled (or, in a
// rollout too dense for lists, each substep's candidates taken), and the queue
// that their contacts are worked out from (physics.rs:241-317).  Shared by the
// differentiable rollouts and the small worlds' step; the general path takes
// the wave scans and the flat rows of cells.
//
// What bounds such a substep is VALU issue and the chain of phases between
// barriers, not memory.  So the grid is fitted when the lists are built and, by
// a world filed every substep, every kFitEvery of them (bodies outside it clamp
// into border cells; any grid gives the same pairs), the scans and reductions
// are DPP chains in registers (a ds_bpermute per step costs the LDS latency six
// times over), and contacts are worked out by all threads from a queue of the
// pairs within reach.
#pragma once

#include "step_common.hpp"

namespace bg {

// ---- wave64 scans and folds in registers ----------------------------------

template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t old, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROWS, 0xf, false);
}

// Inclusive prefix of an associative `op` with identity `id` over the wave's
// lanes (lane 63 ends with the whole wave's fold).  All 64 lanes take part.
template <class Op>
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v, uint32_t id, Op op) {
    v = op(v, dpp_u32<0x111, 0xf>(id, v));  // row_shr 1, 2, 4, 8: prefixes inside rows of 16
    v = op(v, dpp_u32<0x112, 0xf>(id, v));
    v = op(v, dpp_u32<0x114, 0xf>(id, v));
    v = op(v, dpp_u32<0x118, 0xf>(id, v));
    v = op(v, dpp_u32<0x142, 0xa>(id, v));  // lane 15 of rows 0 and 2 to rows 1 and 3
    v = op(v, dpp_u32<0x143, 0xc>(id, v));  // lane 31 to rows 2 and 3
    return v;
}
struct AddU32 {
    __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return a + b; }
};
struct MinU32 {
    __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return min(a, b); }
};
struct MaxU32 {
    __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const { return max(a, b); }
};
struct AddF32 {
    __device__ __forceinline__ uint32_t operator()(uint32_t a, uint32_t b) const {
        return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
    }
};

// Exclusive scan of cnt[0, n) in place by a workgroup of NT threads
// (n <= NT * ITEMS).  Two barriers; red holds NT / 64 words.
template <uint32_t NT, uint32_t ITEMS>
__device__ __forceinline__ void lds_scan(uint32_t* cnt, uint32_t n, uint32_t* red) {
    constexpr uint32_t kNW = NT / BG_WAVE;
    static_assert(kNW <= 16, "one row of wave totals");
    const uint32_t base = threadIdx.x * ITEMS;
    uint32_t v[ITEMS];
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < ITEMS; ++k) {
        v[k] = (base + k < n) ? cnt[base + k] : 0u;
        sum += v[k];
    }
    const uint32_t incl = wave_prefix(sum, 0u, AddU32());
    const uint32_t lane = threadIdx.x & (BG_WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / BG_WAVE));
    if (lane == BG_WAVE - 1) red[wid] = incl;
    __syncthreads();
    uint32_t t = lane < kNW ? red[lane] : 0u;
    t = wave_prefix(t, 0u, AddU32());
    const uint32_t off = wid > 0 ? (uint32_t)__builtin_amdgcn_readlane((int)t, wid - 1) : 0u;
    uint32_t run = off + incl - sum;
#pragma unroll
    for (uint32_t k = 0; k < ITEMS; ++k) {
        if (base + k < n) cnt[base + k] = run;
        run += v[k];
    }
    __syncthreads();
}

// ---- a thread's one or two bodies --------------------------------------------
//
// By selects: an index known only at run time would put the arrays into scratch memory.

template <class T, uint32_t N>
__device__ __forceinline__ T pick(const T (&v)[N], uint32_t j) {
    static_assert(N <= 2, "one select");
    if constexpr (N == 1)
        return v[0];
    else
        return j ? v[1] : v[0];
}
template <uint32_t N>
__device__ __forceinline__ float2 pick(const float2 (&v)[N], uint32_t j) {
    if constexpr (N == 1)
        return v[0];
    else
        return make_float2(j ? v[1].x : v[0].x, j ? v[1].y : v[0].y);
}
template <uint32_t N>
__device__ __forceinline__ void put(float2 (&v)[N], uint32_t j, float2 x) {
    if constexpr (N == 1) {
        v[0] = x;
    } else {
        v[0].x = j ? v[0].x : x.x;
        v[0].y = j ? v[0].y : x.y;
        v[1].x = j ? x.x : v[1].x;
        v[1].y = j ? x.y : v[1].y;
    }
}
template <class T, uint32_t N>
__device__ __forceinline__ void put(T (&v)[N], uint32_t j, T x) {
    if constexpr (N == 1) {
        v[0] = x;
    } else {
        v[0] = j ? v[0] : x;
        v[1] = j ? x : v[1];
    }
}

// ---- the grid -------------------------------------------------------------

constexpr uint32_t kFitEvery = 32;  // substeps between fits of a grid that is filed every substep

struct LdsGrid {
    float ox, oy, inv_cell;
    int32_t nx, ny;
    uint32_t ncells;
    float ex, ey;  // mean of the extra vectors
};

// Sums of one thread's points for the fit, and of an extra vector of some of them.
struct LdsFit {
    float n, sx, sy, sxx, syy, ne, ex, ey;
    uint32_t b0, b1, b2, b3;  // f2ord bounding box
    __device__ __forceinline__ void init() {
        n = sx = sy = sxx = syy = ne = ex = ey = 0.0f;
        b0 = b1 = 0xFFFFFFFFu;
        b2 = b3 = 0u;
    }
    __device__ __forceinline__ void point(float x, float y) {
        if (!finitef(x) || !finitef(y)) return;
        n += 1.0f;
        sx += x;
        sy += y;
        sxx += x * x;
        syy += y * y;
        b0 = min(b0, f2ord(x));
        b1 = min(b1, f2ord(y));
        b2 = max(b2, f2ord(x));
        b3 = max(b3, f2ord(y));
    }
    __device__ __forceinline__ void extra(float x, float y) {
        if (!finitef(x) || !finitef(y)) return;
        ne += 1.0f;
        ex += x;
        ey += y;
    }
};
constexpr uint32_t kFitWords = 12;

// Fits `grid` to the workgroup's points: cells of side `cell` over their
// bounding box, clipped to the centroid +- 3 sigma so that a few bodies thrown
// far away (common after initial overlaps) don't coarsen everyone's cells;
// the cell grows until the box fits `cells`.  Two barriers; red holds
// kFitWords * NT / 64 words and is free again after the second.
template <uint32_t NT>
__device__ __forceinline__ void lds_fit(const LdsFit& f, float cell, uint32_t cells, uint32_t* red, LdsGrid* grid) {
    constexpr uint32_t kNW = NT / BG_WAVE;
    const uint32_t lane = threadIdx.x & (BG_WAVE - 1), wid = threadIdx.x / BG_WAVE;
    auto fold = [](uint32_t (&v)[kFitWords]) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = wave_prefix(v[q], 0u, AddF32());
        v[8] = wave_prefix(v[8], 0xFFFFFFFFu, MinU32());
        v[9] = wave_prefix(v[9], 0xFFFFFFFFu, MinU32());
        v[10] = wave_prefix(v[10], 0u, MaxU32());
        v[11] = wave_prefix(v[11], 0u, MaxU32());
    };
    uint32_t v[kFitWords] = {__float_as_uint(f.n),   __float_as_uint(f.sx), __float_as_uint(f.sy),
                             __float_as_uint(f.sxx), __float_as_uint(f.syy), __float_as_uint(f.ne),
                             __float_as_uint(f.ex),  __float_as_uint(f.ey),  f.b0, f.b1, f.b2, f.b3};
    fold(v);
    if (lane == BG_WAVE - 1) {
#pragma unroll
        for (uint32_t q = 0; q < kFitWords; ++q) red[q * kNW + wid] = v[q];
    }
    __syncthreads();
    if (wid == 0) {
#pragma unroll
        for (uint32_t q = 0; q < kFitWords; ++q) v[q] = lane < kNW ? red[q * kNW + lane] : (q < 8 || q > 9 ? 0u : 0xFFFFFFFFu);
        fold(v);
        if (lane == BG_WAVE - 1) {
            const float n = __uint_as_float(v[0]);
            float minx = 0.0f, miny = 0.0f, maxx = 0.0f, maxy = 0.0f;
            if (!(cell > 0.0f) || !finitef(cell)) cell = 1.0f;
            if (n > 0.0f) {
                minx = ord2f(v[8]);
                miny = ord2f(v[9]);
                maxx = ord2f(v[10]);
                maxy = ord2f(v[11]);
                const float mx = __uint_as_float(v[1]) / n, my = __uint_as_float(v[2]) / n;
                const float dx = 3.0f * sqrtf(fmaxf(__uint_as_float(v[3]) / n - mx * mx, 0.0f)) + cell;
                const float dy = 3.0f * sqrtf(fmaxf(__uint_as_float(v[4]) / n - my * my, 0.0f)) + cell;
                if (finitef(mx) && finitef(dx)) {
                    minx = fmaxf(minx, mx - dx);
                    maxx = fminf(maxx, mx + dx);
                }
                if (finitef(my) && finitef(dy)) {
                    miny = fmaxf(miny, my - dy);
                    maxy = fminf(maxy, my + dy);
                }
            }
            const float ex = fmaxf(maxx - minx, 0.0f), ey = fmaxf(maxy - miny, 0.0f);
            int32_t nx = 1, ny = 1;
            for (;;) {
                const float fx = floorf(ex / cell) + 1.0f, fy = floorf(ey / cell) + 1.0f;
                if (fx <= 65536.0f && fy <= 65536.0f && (uint64_t)fx * (uint64_t)fy <= (uint64_t)cells) {
                    nx = (int32_t)fx;
                    ny = (int32_t)fy;
                    break;
                }
                cell = larger_cell(cell, fx > 65536.0f || fy > 65536.0f ? 16.0f : 1.25f);
                if (!finitef(cell)) break;  // an infinite extent: one cell
            }
            grid->ox = minx;
            grid->oy = miny;
            grid->inv_cell = 1.0f / cell;
            grid->nx = nx;
            grid->ny = ny;
            grid->ncells = (uint32_t)nx * (uint32_t)ny;
            const float ne = __uint_as_float(v[5]);
            grid->ex = ne > 0.0f ? __uint_as_float(v[6]) / ne : 0.0f;
            grid->ey = ne > 0.0f ? __uint_as_float(v[7]) / ne : 0.0f;
        }
    }
    __syncthreads();
}

// The grid's fields, the same in every lane, as scalars.
__device__ __forceinline__ LdsGrid lds_grid_uniform(const LdsGrid& g) {
    auto f = [](float v) { return __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(v))); };
    LdsGrid u;
    u.ox = f(g.ox);
    u.oy = f(g.oy);
    u.inv_cell = f(g.inv_cell);
    u.nx = __builtin_amdgcn_readfirstlane(g.nx);
    u.ny = __builtin_amdgcn_readfirstlane(g.ny);
    u.ncells = (uint32_t)__builtin_amdgcn_readfirstlane((int)g.ncells);
    u.ex = f(g.ex);
    u.ey = f(g.ey);
    return u;
}

__device__ __forceinline__ uint32_t lds_cell(const LdsGrid& g, float x, float y) {
    return (uint32_t)cell_coord(y, g.oy, g.inv_cell, g.ny) * (uint32_t)g.nx +
           (uint32_t)cell_coord(x, g.ox, g.inv_cell, g.nx);
}

// ---- contacts ----------------------------------------------------------------
//
// Three phases with a barrier between them.  Mark: each body puts its partners
// within reach into a queue.  Correct: a thread takes one queued pair, whoever's
// it is, and works out its correction (a root and three divides, about 200
// instructions): with one contact among ten bodies a wave that corrected its own
// would run that code once or twice for each of its bodies, almost all lanes idle.
// Sum: each body adds its corrections in ascending partner index.

constexpr int kLdsRows = 3;        // grid rows of a flat candidate list (a query of cells of 2 r_max rarely spans 4)
constexpr uint32_t kLdsFlat = 64;  // candidates of a flat list (one 64-bit mask)
constexpr uint32_t kLdsRecPad = 4;
constexpr uint32_t kNoPair = 0xFFFFFFFFu;

// Cells of the square of half-width Q around (x, y); the whole grid when it is not finite.
struct LdsRect {
    int32_t cx0, cx1, cy0, cy1;
};
__device__ __forceinline__ LdsRect lds_rect(const LdsGrid& g, float x, float y, float Q) {
    const float R = Q + (1e-5f * (fabsf(x) + fabsf(y) + Q) + 1e-6f);
    LdsRect c = {0, g.nx - 1, 0, g.ny - 1};
    if (R < 1e30f && finitef(x) && finitef(y)) {
        c.cx0 = cell_coord(x - R, g.ox, g.inv_cell, g.nx);
        c.cx1 = cell_coord(x + R, g.ox, g.inv_cell, g.nx);
        c.cy0 = cell_coord(y - R, g.oy, g.inv_cell, g.ny);
        c.cy1 = cell_coord(y + R, g.oy, g.inv_cell, g.ny);
    }
    return c;
}

// A body's pairs in the queue: `n` entries from `first`, or (direct: no room for them) its
// contacts are left to the caller.
struct LdsPairs {
    uint32_t first, n;
    bool direct;
};

// Queue a body's marked candidates (bit i: other(i)), a body a lane, by whole waves.  *count
// was zero before the phase; entries from CAP on are not written, and a body that has some
// there is left to the caller.
template <uint32_t CAP, class Other>
__device__ __forceinline__ LdsPairs lds_queue(uint64_t marked, uint32_t own, uint32_t* entries, uint32_t* count,
                                              Other&& other) {
    LdsPairs pr;
    pr.n = (uint32_t)__popcll(marked);
    pr.direct = false;
    const uint32_t incl = wave_prefix(pr.n, 0u, AddU32());
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, BG_WAVE - 1);
    uint32_t at = 0;
    if (total > 0) {
        if ((threadIdx.x & (BG_WAVE - 1)) == 0) at = atomicAdd(count, total);
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
    }
    pr.first = at + incl - pr.n;
    const bool fits = pr.first + pr.n <= CAP;
    for (uint32_t e = pr.first; marked != 0; ++e) {
        const uint32_t i = (uint32_t)__builtin_ctzll(marked);
        marked &= marked - 1;
        if (e < CAP) entries[e] = fits ? (own << 16) | other(i) : kNoPair;
    }
    if (!fits) {
        pr.direct = true;
        pr.n = 0;
    }
    return pr;
}

// The records of up to kLdsRows rows of cells as one flat list: entry i is record base + i, plus
// step1 from end0 on (the second row), plus step2 from end1 on (all modulo 2^32).  (Sums,
// because a select between two variables here is compiled to a load through a selected address.)
struct LdsRows {
    uint32_t base, end0, step1, end1, step2, n;
    bool flat;  // the rows and records fit (else n is 0)
    __device__ __forceinline__ uint32_t slot(uint32_t i) const {
        return (i >= end0 ? step1 : 0u) + (i >= end1 ? step2 : 0u) + (base + i);
    }
};
// The cells of `c` in a grid of nx columns (neither past 65,536) whose records start at start[cell].
__device__ __forceinline__ LdsRows flat_rows(const uint32_t* start, uint32_t nx, const LdsRect& c) {
    LdsRows l;
    const uint32_t row0 = __umul24((uint32_t)c.cy0, nx), last = __umul24((uint32_t)c.cy1, nx);
    const uint32_t row1 = min(row0 + nx, last), row2 = min(row1 + nx, last);
    const uint32_t* s0 = start + c.cx0;
    const uint32_t* s1 = start + c.cx1 + 1;
    const uint32_t lo0 = s0[row0], hi0 = s1[row0], lo1 = s0[row1], hi1 = s1[row1], lo2 = s0[row2], hi2 = s1[row2];
    const int32_t rows = c.cy1 - c.cy0 + 1;
    l.base = lo0;
    l.end0 = hi0 - lo0;
    l.step1 = lo1 - hi0;
    l.end1 = l.end0 + (rows > 1 ? hi1 - lo1 : 0u);
    l.step2 = (lo2 - l.end1) - (lo1 - l.end0);
    l.n = l.end1 + (rows > 2 ? hi2 - lo2 : 0u);
    l.flat = rows <= kLdsRows && l.n <= kLdsFlat;
    if (!l.flat) l.n = 0;
    static_assert(kLdsRows == 3, "the rows above");
    return l;
}
__device__ __forceinline__ LdsRows lds_rows(const LdsGrid& g, const uint32_t* start, bool active, float2 xy, float Q) {
    LdsRows l = {0, 0, 0, 0, 0, 0, false};
    if (active) l = flat_rows(start, (uint32_t)g.nx, lds_rect(g, xy.x, xy.y, Q));
    return l;
}

// The entries of a flat list that near(slot, record) accepts, one bit each.  (Past the last one it
// reads up to three records further -- rec has kLdsRecPad records of room -- and drops their bits.)
template <class Near>
__device__ __forceinline__ uint64_t lds_near(const LdsRows& l, const float4* rec, Near&& near) {
    uint32_t near_lo = 0, near_hi = 0;
    auto four = [&](uint32_t f) -> uint32_t {
        float4 sb[4];
        uint32_t t[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            t[u] = l.slot(f + u);
            sb[u] = rec[t[u]];
        }
        uint32_t bits = 0;
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) bits |= near(t[u], sb[u]) ? 1u << u : 0u;
        return bits;
    };
    for (uint32_t f = 0; f < min(l.n, 32u); f += 4) near_lo |= four(f) << f;
    for (uint32_t f = 32; f < l.n; f += 4) near_hi |= four(f) << (f - 32u);
    if (l.n < 32u) near_lo &= (1u << l.n) - 1u;
    if (l.n < 64u) near_hi &= l.n > 32u ? (1u << (l.n - 32u)) - 1u : 0u;
    return ((uint64_t)near_hi << 32) | near_lo;
}

// One pair: its contact (physics.rs:264-300) from the side of the body `own`.
// A is the body of the higher index (local order is arena order).
struct LdsContact {
    float2 c;     // correction of the body's position
    bool hit;     // a contact
    bool pushed;  // took the push-out branch, folded into the correction by the pair rule
    bool nan;     // its normal is not a number
};
__device__ __forceinline__ LdsContact lds_correction(const float4 own, const float4 other, float m_own, float m_other,
                                                     bool is_a, bool sensor) {
    LdsContact r = {make_float2(0.0f, 0.0f), false, false, false};
    const float dx = own.x - other.x, dy = own.y - other.y;
    const float rs = own.z + other.z;
    const float dot = dx * dx + dy * dy;
    if (dot > (rs * rs) * 1.00000095367431640625f) return r;
    float dist = sqrtf(dot);
    if (!(dist < rs)) return r;
    r.hit = true;
    float ax = is_a ? dx : -dx;
    const float ay = is_a ? dy : -dy;
    float px = 0.0f, py = 0.0f;
    r.pushed = dist < 1e-6f;
    if (r.pushed) {
        ax = ax + 0.02f;
        dist = vlen(ax, ay);
        px = is_a ? 0.01f : -0.01f;
        py = is_a ? 0.0f : -0.0f;
    }
    if (sensor) {
        r.c = make_float2(px, py);
        return r;
    }
    const float mA = is_a ? m_own : m_other, mB = is_a ? m_other : m_own;
    const float ratio = 1.0f - mA / (mA + mB);
    const float nx = ax / dist, ny = ay / dist;
    r.nan = nx != nx || ny != ny;
    const float delta = rs - dist;
    const float kk = is_a ? ratio * delta : (1.0f - ratio) * delta;
    r.c.x = is_a ? kk * nx : -(kk * nx);
    r.c.y = is_a ? kk * ny : -(kk * ny);
    if (r.pushed) {
        r.c.x = px + r.c.x;
        r.c.y = py + r.c.y;
    }
    return r;
}

// Sum phase: f(k, partner, correction) over the body's contacts in ascending partner index.
template <class F>
__device__ __forceinline__ uint32_t lds_sum(const LdsPairs& pr, const uint32_t* entries, const float2* res, F&& f) {
    uint32_t k = 0;
    for (uint32_t next = 0; k < pr.n; ++k) {
        uint32_t best = kNoPair, at = 0;
        for (uint32_t e = pr.first; e < pr.first + pr.n; ++e) {
            const uint32_t key = entries[e];
            if (key >= next && key < best) {
                best = key;
                at = e;
            }
        }
        if (best == kNoPair) break;
        f(k, best, res[at]);
        next = best + 1u;
    }
    return k;
}

}  // namespace bg
