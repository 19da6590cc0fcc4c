// One-sided direct sum in blocks of 16 targets, shared by the single-system
// step (ds_kernels.hip) and the batch (batch_kernels.hip).
//
// lane = 16 * slot + stream: a wave holds 16 targets, four per lane (t = 4 *
// slot + r), and sixteen sources at a time, one per stream.  A target's sum is
// split over 16 roles of 16 streams: role w, stream s takes the sources
// (16 k + w) * 16 + s, k = 0, 1, ...; each stream adds its sources in order, a
// role's streams are added by exchange with stream ^ 15, ^ 7, ^ 2 and ^ 1, and
// the roles in order.  The single-system step runs the roles on the 16 waves
// of a workgroup and adds them through LDS; the batch runs them one after
// another on one wave: the same additions in the same order.
#pragma once

#include "internal.hpp"
#include "lane_ops.hpp"

namespace gsim {

constexpr uint32_t kDsRoles = 16;       // waves of a workgroup

struct DsSource {
    float x, y, m;
};

__device__ __forceinline__ DsSource ds_source(const float2 *__restrict__ pos,
                                              const float *__restrict__ mass, uint32_t j) {
    const float2 p = pos[j];
    return DsSource{p.x, p.y, mass[j]};
}

// kRcp: 1/r2 from v_rcp_f32 instead of inv*inv.
template <bool kRcp>
__device__ __forceinline__ void ds_add(const DsSource &q, const float (&tx)[4],
                                       const float (&ty)[4], float eps2, float (&ax)[4],
                                       float (&ay)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float dx = q.x - tx[r], dy = q.y - ty[r];
        const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, eps2));
        const float inv = __builtin_amdgcn_rsqf(r2);
        const float inv2 = kRcp ? __builtin_amdgcn_rcpf(r2) : inv * inv;
        const float t = (q.m * inv) * inv2;
        ax[r] = __builtin_fmaf(dx, t, ax[r]);
        ay[r] = __builtin_fmaf(dy, t, ay[r]);
        __builtin_amdgcn_sched_barrier(0);  // pairs in sequence issue faster than interleaved
    }
}

// The sum over a slot's 16 streams of target 4 * slot + (stream >> 2).
__device__ __forceinline__ float ds_sum_streams(const float (&a)[4], uint32_t lane) {
    const bool up = (lane & 8u) != 0, u2 = (lane & 4u) != 0;
    const float b0 = (up ? a[2] : a[0]) + dpp<kDppXor15>(up ? a[0] : a[2]);
    const float b1 = (up ? a[3] : a[1]) + dpp<kDppXor15>(up ? a[1] : a[3]);
    const float c = (u2 ? b1 : b0) + dpp<kDppXor7>(u2 ? b0 : b1);
    const float d = c + dpp<kDppXor2>(c);
    return d + dpp<kDppXor1>(d);
}

}  // namespace gsim
