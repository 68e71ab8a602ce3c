// lds_grid.hpp -- contacts of one world inside one workgroup: its bodies'
// snapshot filed by cell in LDS every substep, and the contact pass of one
// body over it (physics.rs:241-317).  Shared by the differentiable rollouts
// and the persistent step.
//
// What bounds such a substep is VALU issue and the chain of phases between
// barriers, not memory.  So the grid is fitted once every kFitEvery substeps
// (bodies outside it clamp into border cells; any grid gives the same pairs),
// the scans and reductions are DPP chains in registers (a ds_bpermute per
// step costs the LDS latency six times over), and a body first marks its
// candidates within reach in a bit mask with about 20 instructions each and
// takes the exact test and the correction (three divides and a root, about
// 130 instructions) for marked ones only.
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

// ---- the grid -------------------------------------------------------------

constexpr uint32_t kFitEvery = 32;  // substeps between fits of the grid to the bodies

struct LdsGrid {
    float ox, oy, inv_cell;
    int32_t nx, ny;
    uint32_t ncells;
};

// Sums of one thread's points for the fit.
struct LdsFit {
    float n, sx, sy, sxx, syy;
    uint32_t b0, b1, b2, b3;  // f2ord bounding box
    __device__ __forceinline__ void init() {
        n = sx = sy = sxx = syy = 0.0f;
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
};
constexpr uint32_t kFitWords = 9;

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
        for (int q = 0; q < 5; ++q) v[q] = wave_prefix(v[q], 0u, AddF32());
        v[5] = wave_prefix(v[5], 0xFFFFFFFFu, MinU32());
        v[6] = wave_prefix(v[6], 0xFFFFFFFFu, MinU32());
        v[7] = wave_prefix(v[7], 0u, MaxU32());
        v[8] = wave_prefix(v[8], 0u, MaxU32());
    };
    uint32_t v[kFitWords] = {__float_as_uint(f.n),   __float_as_uint(f.sx), __float_as_uint(f.sy),
                             __float_as_uint(f.sxx), __float_as_uint(f.syy), f.b0, f.b1, f.b2, f.b3};
    fold(v);
    if (lane == BG_WAVE - 1) {
#pragma unroll
        for (uint32_t q = 0; q < kFitWords; ++q) red[q * kNW + wid] = v[q];
    }
    __syncthreads();
    if (wid == 0) {
#pragma unroll
        for (uint32_t q = 0; q < kFitWords; ++q) v[q] = lane < kNW ? red[q * kNW + lane] : (q < 5 || q > 6 ? 0u : 0xFFFFFFFFu);
        fold(v);
        if (lane == BG_WAVE - 1) {
            const float n = __uint_as_float(v[0]);
            float minx = 0.0f, miny = 0.0f, maxx = 0.0f, maxy = 0.0f;
            if (!(cell > 0.0f) || !finitef(cell)) cell = 1.0f;
            if (n > 0.0f) {
                minx = ord2f(v[5]);
                miny = ord2f(v[6]);
                maxx = ord2f(v[7]);
                maxy = ord2f(v[8]);
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
                cell = cell * (fx > 65536.0f || fy > 65536.0f ? 16.0f : 1.25f);
                if (!finitef(cell)) break;  // an infinite extent: one cell
            }
            grid->ox = minx;
            grid->oy = miny;
            grid->inv_cell = 1.0f / cell;
            grid->nx = nx;
            grid->ny = ny;
            grid->ncells = (uint32_t)nx * (uint32_t)ny;
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
    return u;
}

__device__ __forceinline__ uint32_t lds_cell(const LdsGrid& g, float x, float y) {
    return (uint32_t)cell_coord(y, g.oy, g.inv_cell, g.ny) * (uint32_t)g.nx +
           (uint32_t)cell_coord(x, g.ox, g.inv_cell, g.nx);
}

// ---- one body's contacts ----------------------------------------------------

constexpr int kLdsRows = 3;          // grid rows of a flat candidate list (a query of cells of 2 r_max rarely spans 4)
constexpr uint32_t kLdsFlat = 64;    // candidates of a flat list (one 64-bit mask)

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

// The records of those cells, as one flat list where they are few enough.
struct LdsQuery {
    uint32_t end[kLdsRows - 1];  // flat end of each row but the last
    uint32_t base[kLdsRows];     // record of flat index i in row r: base[r] + i (modulo 2^32)
    uint32_t n;
    bool flat;
    __device__ __forceinline__ uint32_t slot(uint32_t i) const {
        uint32_t b = base[0];
#pragma unroll
        for (int r = 1; r < kLdsRows; ++r) b = i >= end[r - 1] ? base[r] : b;
        return b + i;
    }
};

__device__ __forceinline__ LdsQuery lds_query(const LdsGrid& g, const uint32_t* start, float x, float y, float Q) {
    const LdsRect c = lds_rect(g, x, y, Q);
    LdsQuery q;
    q.n = 0;
#pragma unroll
    for (int r = 0; r < kLdsRows; ++r) {
        const int32_t cy = c.cy0 + r;
        uint32_t lo = 0, hi = 0;
        if (cy <= c.cy1) {
            const uint32_t row = (uint32_t)cy * (uint32_t)g.nx;
            lo = start[row + (uint32_t)c.cx0];
            hi = start[row + (uint32_t)c.cx1 + 1u];
        }
        q.base[r] = lo - q.n;
        q.n += hi - lo;
        if (r + 1 < kLdsRows) q.end[r] = q.n;
    }
    q.flat = c.cy1 - c.cy0 < kLdsRows && q.n <= kLdsFlat;
    return q;
}

// Contacts of body `li` (snapshot xy, radius r, mass m) with the records
// rec[] = (x, y, radius, bits(local index)) of the grid, summed into `p` in
// ascending partner index.  A is the body of the higher index (local order is
// arena order).  `mass(lj)` is a partner's mass, `skip(lj)` drops a candidate
// (interaction groups), `sensor(lj)` keeps a contact out of the sums, and
// `hit(lj, isA, pushed, nan)` is called once for each contact.  Returns their
// number; L ends with the K smallest partners' corrections.
template <int K, class Mass, class Skip, class Sensor, class Hit>
__device__ __forceinline__ uint32_t lds_contacts(const LdsGrid& g, const uint32_t* start, const float4* rec, float2 xy,
                                                 float r, float m, uint32_t li, float rmax, float2& p,
                                                 ContactList<K, uint32_t>& L, Mass&& mass, Skip&& skip,
                                                 Sensor&& sensor, Hit&& hit) {
    const LdsQuery q = lds_query(g, start, xy.x, xy.y, r + rmax);
    uint32_t near_lo = 0, near_hi = 0;
    auto mark = [&](uint32_t f) -> uint32_t {  // four candidates
        float4 sb[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) sb[u] = rec[q.slot(min(f + u, q.n - 1u))];
        uint32_t bits = 0;
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const float dx = xy.x - sb[u].x, dy = xy.y - sb[u].y;
            const float rs = r + sb[u].z;
            const bool cand = f + u < q.n && __float_as_uint(sb[u].w) != li &&
                              !(dx * dx + dy * dy > (rs * rs) * 1.00000095367431640625f);
            bits |= cand ? 1u << u : 0u;
        }
        return bits;
    };
    if (q.flat) {
        for (uint32_t f = 0; f < min(q.n, 32u); f += 4) near_lo |= mark(f) << f;
        for (uint32_t f = 32; f < q.n; f += 4) near_hi |= mark(f) << (f - 32u);
    }
    // the reference predicate (physics.rs:264-269) and, for a contact, its correction
    auto test = [&](const float4 sb, auto&& sink) {
        const uint32_t lj = __float_as_uint(sb.w);
        if (lj == li || skip(lj)) return;
        const bool isA = li > lj;
        const float dx = xy.x - sb.x, dy = xy.y - sb.y;
        const float rs = r + sb.z;
        const float dot = dx * dx + dy * dy;
        if (dot > (rs * rs) * 1.00000095367431640625f) return;
        const float dist = sqrtf(dot);
        if (!(dist < rs)) return;
        sink(lj, isA, isA ? dx : -dx, isA ? dy : -dy, dist, rs);
    };
    auto enumerate = [&](auto&& sink) {
        if (q.flat) {
            uint64_t mm = ((uint64_t)near_hi << 32) | near_lo;
            while (mm != 0) {
                const uint32_t i = (uint32_t)__builtin_ctzll(mm);
                mm &= mm - 1;
                test(rec[q.slot(i)], sink);
            }
        } else {
            const LdsRect c = lds_rect(g, xy.x, xy.y, r + rmax);
            for (int32_t cy = c.cy0; cy <= c.cy1; ++cy) {
                const uint32_t row = (uint32_t)cy * (uint32_t)g.nx;
                const uint32_t t1 = start[row + (uint32_t)c.cx1 + 1u];
                for (uint32_t t = start[row + (uint32_t)c.cx0]; t < t1; ++t) test(rec[t], sink);
            }
        }
    };
    // correction on this body from one pair (physics.rs:270-300); a push-out is folded into
    // the same entry by the pair rule
    auto correction = [&](auto&& put, auto&& once, uint32_t lj, bool isA, float ax, float ay, float dist, float rs) {
        float px = 0.0f, py = 0.0f;
        const bool pushed = dist < 1e-6f;
        if (pushed) {
            ax = ax + 0.02f;
            dist = vlen(ax, ay);
            px = isA ? 0.01f : -0.01f;
            py = isA ? 0.0f : -0.0f;
        }
        if (sensor(lj)) {
            once(pushed, false);
            if (pushed) put(lj, px, py);
            return;
        }
        const float mpart = mass(lj);
        const float mA = isA ? m : mpart, mB = isA ? mpart : m;
        const float ratio = 1.0f - mA / (mA + mB);
        const float nx = ax / dist, ny = ay / dist;
        once(pushed, nx != nx || ny != ny);
        const float delta = rs - dist;
        float cx, cy;
        if (isA) {
            const float kk = ratio * delta;
            cx = kk * nx;
            cy = kk * ny;
        } else {
            const float kk = (1.0f - ratio) * delta;
            cx = -(kk * nx);
            cy = -(kk * ny);
        }
        if (pushed) {
            cx = px + cx;
            cy = py + cy;
        }
        put(lj, cx, cy);
    };
    L.init();
    uint32_t found = 0;
    enumerate([&](uint32_t lj, bool isA, float ax, float ay, float dist, float rs) {
        ++found;
        correction([&](uint32_t kk, float x, float y) { L.add(kk, x, y); },
                   [&](bool pushed, bool nan) { hit(lj, isA, pushed, nan); }, lj, isA, ax, ay, dist, rs);
    });
    if (L.n > 0) {
        uint32_t last = L.apply(p);
        uint32_t done = L.n < (uint32_t)K ? L.n : (uint32_t)K;
        while (done < L.n) {  // more than K: next partner by selection, same order
            uint32_t best = 0xFFFFFFFFu;
            float bx = 0.0f, by = 0.0f;
            enumerate([&](uint32_t lj, bool isA, float ax, float ay, float dist, float rs) {
                correction(
                    [&](uint32_t kk, float x, float y) {
                        if (kk > last && kk < best) {
                            best = kk;
                            bx = x;
                            by = y;
                        }
                    },
                    [](bool, bool) {}, lj, isA, ax, ay, dist, rs);
            });
            if (best == 0xFFFFFFFFu) break;
            p.x = p.x + bx;
            p.y = p.y + by;
            last = best;
            ++done;
        }
    }
    return found;
}

}  // namespace bg
