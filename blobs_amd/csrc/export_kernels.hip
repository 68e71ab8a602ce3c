// export_kernels.hip -- a world's state for the host, in dense (arena
// iteration) order.
//
// On the sphere path slot k holds dense body id(k), so the records are
// scattered by id here instead of on the host, into arenas whose entries span
// cache lines.  Bound by the host link.  Read-back of a world, before (six
// copies to pageable memory and the host mirror) and now: 1,048,576 bodies
// 129 -> 1.7 ms, 65,536 3.2 -> 0.16 ms, 1,288 146 -> 37 us, 100 108 -> 27 us.
#include <algorithm>

#include "device_state.hpp"
#include "step_common.hpp"

namespace bg {

namespace {

__global__ __launch_bounds__(kThreads) void k_export_sphere(const float4* __restrict__ pp,
                                                            const float4* __restrict__ snap,
                                                            const float2* __restrict__ vel,
                                                            const float2* __restrict__ rw,
                                                            const float* __restrict__ wold_dt, uint32_t n_worlds,
                                                            uint32_t nb, uint32_t id_mask, ExportOut o) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (o.old_dt)
        for (uint32_t w = k; w < n_worlds; w += gridDim.x * blockDim.x) o.old_dt[w] = wold_dt[w];
    if (k >= nb) return;
    const float4 sn = snap[k];
    const uint32_t id = __float_as_uint(sn.w) & id_mask;
    if (id >= nb) return;  // ids are a permutation of [0, nb)
    if (o.pos || o.pos_old) {
        const float4 p = pp[k];
        if (o.pos) o.pos[id] = make_float2(p.x, p.y);
        if (o.pos_old) o.pos_old[id] = make_float2(p.z, p.w);
    }
    if (o.vel) o.vel[id] = vel[k];
    if (o.rot || o.omega) {
        const float2 r = rw[k];
        if (o.rot) o.rot[id] = r.x;
        if (o.omega) o.omega[id] = r.y;
    }
    if (o.col_pos) o.col_pos[id] = make_float2(sn.x, sn.y);
}

__global__ __launch_bounds__(kThreads) void k_export_general(BodyArrays b, const float2* __restrict__ abs, uint32_t nb,
                                                             uint32_t nc, const StepAccum* accum, ExportOut o) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0 && o.old_dt) *o.old_dt = accum->old_dt;
    if (k < nb) {
        if (o.pos) o.pos[k] = b.pos[k];
        if (o.pos_old) o.pos_old[k] = b.pos_old[k];
        if (o.vel) o.vel[k] = b.vel[k];
        if (o.rot) o.rot[k] = b.rot[k];
        if (o.omega) o.omega[k] = b.omega[k];
    }
    if (k < nc && o.col_pos) o.col_pos[k] = abs[k];
}

}  // namespace

hipError_t launch_export(const DeviceWorld& d, bool sphere, uint32_t id_mask, const ExportOut& out) {
    const uint32_t n = std::max<uint32_t>(std::max(d.nb, d.nc), 1);
    if (sphere)
        k_export_sphere<<<div_up(n, kThreads), kThreads, 0, d.stream>>>(d.s.pp, d.s.snap, d.s.vel, d.s.rw, d.wold_dt,
                                                                       d.n_worlds, d.nb, id_mask, out);
    else
        k_export_general<<<div_up(n, kThreads), kThreads, 0, d.stream>>>(d.b, d.c.abs, d.nb, d.nc, d.accum, out);
    return hipGetLastError();
}

}  // namespace bg
