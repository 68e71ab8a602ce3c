// step_common.hpp -- device helpers shared by the general and the fused
// sphere substep kernels (compiled with -ffp-contract=off, like every kernel
// source here: the reference never fuses a*b+c).
#pragma once

#include <float.h>

#include "common.hpp"
#include "device_state.hpp"

namespace bg {

constexpr int kThreads = 256;

inline uint32_t div_up(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// Workgroups are dispatched round-robin over the 8 XCDs of an MI355X, each
// with its own L2.  Renumbering them so that every XCD gets one contiguous
// range of slots keeps a body's grid neighbours (same and adjacent cell
// rows) in the L2 of the XCD that reads them.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t n) {
    const uint32_t q = n / 8u, r = n % 8u;
    const uint32_t x = b % 8u, i = b / 8u;
    return x * q + (x < r ? x : r) + i;
}

// ---- sorted register list of contact corrections -------------------------
// Keeps the K smallest keys in ascending order (unrolled insertion with
// compile-time indices, so it stays in VGPRs); `n` counts every insertion.
template <int K, typename Key>
struct ContactList {
    Key key[K];
    float cx[K], cy[K];
    uint32_t n;
    __device__ __forceinline__ void init() {
        n = 0;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            key[i] = (Key)~(Key)0;
            cx[i] = 0.0f;
            cy[i] = 0.0f;
        }
    }
    __device__ __forceinline__ void add(Key k, float x, float y) {
        Key ck = k;
        float ccx = x, ccy = y;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            bool sw = ck < key[i];
            Key tk = key[i];
            float tx = cx[i], ty = cy[i];
            key[i] = sw ? ck : tk;
            cx[i] = sw ? ccx : tx;
            cy[i] = sw ? ccy : ty;
            ck = sw ? tk : ck;
            ccx = sw ? tx : ccx;
            ccy = sw ? ty : ccy;
        }
        ++n;
    }
    // Adds the stored corrections in key order; returns the last key applied.
    __device__ __forceinline__ Key apply(float2& p) const {
        Key last = 0;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            if ((uint32_t)i < n) {
                p.x = p.x + cx[i];
                p.y = p.y + cy[i];
                last = key[i];
            }
        }
        return last;
    }
};

// Q padded for the rounding of cell coordinates.
__device__ __forceinline__ float stencil_reach(float2 q, float Q) {
    return Q + (1e-5f * (fabsf(q.x) + fabsf(q.y) + Q) + 1e-6f);
}

// Visit every slot in the cells overlapping the square of half-width Q
// around (qx, qy), in slot order, four at a time: visit(t, r, nv) gets slots
// t .. t+nv-1 (nv in 1..4) with their records r[0..nv-1] (loaded together,
// so their loads overlap).  Cell coordinates are monotone in x, so the
// visited set is a superset of all snapshots within distance Q of the query
// point.
template <class F>
__device__ __forceinline__ void scan_stencil(const GridParams& g, const uint32_t* __restrict__ cell_start, uint32_t n,
                                             const float4* __restrict__ rec, float qx, float qy, float Q, F&& visit) {
    const float R = stencil_reach(make_float2(qx, qy), Q);
    int32_t cx0, cx1, cy0, cy1;
    if (R < 1e30f && finitef(qx) && finitef(qy)) {
        cx0 = cell_coord(qx - R, g.ox, g.inv_cell, g.nx);
        cx1 = cell_coord(qx + R, g.ox, g.inv_cell, g.nx);
        cy0 = cell_coord(qy - R, g.oy, g.inv_cell, g.ny);
        cy1 = cell_coord(qy + R, g.oy, g.inv_cell, g.ny);
    } else {
        cx0 = 0;
        cx1 = g.nx - 1;
        cy0 = 0;
        cy1 = g.ny - 1;
    }
    for (int32_t cy = cy0; cy <= cy1; ++cy) {
        uint32_t row = (uint32_t)cy * (uint32_t)g.nx;
        uint32_t t0 = cell_start[row + (uint32_t)cx0];
        uint32_t t1 = cell_start[row + (uint32_t)cx1 + 1u];
        t1 = t1 < n ? t1 : n;  // cell_start is a monotone table in [0, n]
        for (uint32_t t = t0; t < t1; t += 4) {
            float4 r[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) r[u] = rec[min(t + u, t1 - 1u)];
            visit(t, r, t1 - t < 4u ? t1 - t : 4u);
        }
    }
}

// Only blocks that extend the running extremum issue an atomic (a relaxed
// read first): thousands of blocks hitting one word serialize otherwise.
__device__ __forceinline__ void atomic_max_if_greater(uint32_t* p, uint32_t v) {
    if (v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p, v);
}
__device__ __forceinline__ void atomic_min_if_less(uint32_t* p, uint32_t v) {
    if (v < __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(p, v);
}

// ---- Verlet update of one body, physics.rs:326-358 -----------------------
struct BodyState {
    float2 p, po, vel;
    float rot, omega;
};

__device__ __forceinline__ void verlet_dynamic(BodyState& s, float2 acc, float torque_over_inertia, bool has_vreq,
                                               float2 vreq, float h, float ratio) {
    if (has_vreq) {  // :334-336
        s.po.x = s.p.x - vreq.x * h;
        s.po.y = s.p.y - vreq.y * h;
    }
    float dx = (s.p.x - s.po.x) * ratio;  // :338
    float dy = (s.p.y - s.po.y) * ratio;
    s.po = s.p;                                    // :343
    s.p.x = s.p.x + (dx + (acc.x * h) * h);        // :344
    s.p.y = s.p.y + (dy + (acc.y * h) * h);
    s.omega = s.omega + torque_over_inertia * h;   // :346
    s.rot = s.rot + s.omega * h;                   // :349
    s.vel.x = dx / h;                              // :357
    s.vel.y = dy / h;
}

// Position part of one fixed joint (physics.rs:434-460) on body positions pa,
// pb; the axis d = wb - wa goes to (dx, dy).  Returns false for coincident
// anchors, which the reference skips.
__device__ __forceinline__ bool joint_positions(float2& pa, float2& pb, float2 an_a, float2 an_b, float jdist,
                                                float4 jm, bool sa, bool sb, float& dx, float& dy,
                                                uint32_t& flags) {
    float wax = pa.x + an_a.x, way = pa.y + an_a.y;
    float wbx = pb.x + an_b.x, wby = pb.y + an_b.y;
    dx = wbx - wax;
    dy = wby - way;
    float dist = vlen(dx, dy);
    if (dist < 1e-6f) return false;
    float off_by = dist - jdist;
    float cx = (off_by * dx) / dist, cy = (off_by * dy) / dist;
    if (jm.w == 0.0f) flags |= ERR_JOINT_MASS;
    const float ims = jm.x;
    if (sa) {
        pb.x = pb.x - ims * cx;
        pb.y = pb.y - ims * cy;
    } else if (sb) {
        pa.x = pa.x + ims * cx;
        pa.y = pa.y + ims * cy;
    } else {
        const float ratio = jm.y, rbm = jm.z;
        pa.x = pa.x + ratio * cx;
        pa.y = pa.y + ratio * cy;
        pb.x = pb.x - rbm * cx;
        pb.y = pb.y - rbm * cy;
    }
    return true;
}

// Circle constraints, physics.rs:377-395 (centre clamp, static bodies too).
__device__ __forceinline__ void apply_constraints(float2& p, const float2* __restrict__ con_pos,
                                                  const float* __restrict__ con_r, uint32_t nk) {
    for (uint32_t k = 0; k < nk; ++k) {
        float2 c = con_pos[k];
        float r = con_r[k];
        float tx = p.x - c.x, ty = p.y - c.y;
        float dist = vlen(tx, ty);
        if (dist > r) {
            float nx = tx / dist, ny = ty / dist;
            p.x = c.x + nx * r;
            p.y = c.y + ny * r;
        }
    }
}

// ============================================================ broadphase

__device__ __forceinline__ GridParams grid_from_bbox(const uint32_t* bb, float cell, uint32_t cells_cap) {
    GridParams g;
    float minx = ord2f(bb[0]), miny = ord2f(bb[1]), maxx = ord2f(bb[2]), maxy = ord2f(bb[3]);
    if (!(minx <= maxx) || !(miny <= maxy) || !finitef(minx) || !finitef(maxx) || !finitef(miny) ||
        !finitef(maxy)) {
        minx = miny = 0.0f;
        maxx = maxy = 0.0f;
    }
    if (!(cell > 0.0f) || !finitef(cell)) cell = 1.0f;
    const float ex = fminf(maxx - minx, 3.0e38f), ey = fminf(maxy - miny, 3.0e38f);
    // A box of more cells than there are takes the smallest cell that fits, not the next double:
    // the crowded middle of a scene that flies apart pays for each needless half.  512 worlds of 1.5M
    // bodies, 60 steps 51.1 -> 41.1 ms (fewer bodies are without a list), 50,021 bodies, 30 steps 3.82 ->
    // 3.56 ms, 294,249 colliders, 8 steps 9.30 -> 8.95-9.02 ms (its scan covers more cells; clipped 8.28).
    bool fitted = false;
    int32_t nx, ny;
    for (;;) {
        float fx = floorf(ex / cell) + 1.0f, fy = floorf(ey / cell) + 1.0f;
        if (fx <= 65536.0f && fy <= 65536.0f && (uint64_t)fx * (uint64_t)fy <= (uint64_t)cells_cap) {
            nx = (int32_t)fx;
            ny = (int32_t)fy;
            break;
        }
        if (fitted) {
            cell = larger_cell(cell, 1.0625f);  // the partial cells at the edges
        } else {
            const float cap = (float)min(cells_cap, 1u << 30);
            cell = fmaxf(cell, fmaxf(sqrtf(ex) * (sqrtf(ey) / sqrtf(cap)), fmaxf(ex, ey) / fminf(65536.0f, cap)));
            fitted = true;
        }
    }
    g.ox = minx;
    g.oy = miny;
    g.cell = cell;
    g.inv_cell = 1.0f / cell;
    g.nx = nx;
    g.ny = ny;
    g.ncells = (uint32_t)nx * (uint32_t)ny;
    g.pad = 0;
    return g;
}


}  // namespace bg
