// One-sided direct sum in blocks of 16 targets, shared by the single-system
// step (ds_kernels.hip) and the batch (batch_kernels.hip).
//
// lane = 16 * slot + stream: a wave holds 16 targets, four per lane (t = 4 *
// slot + r), and sixteen sources at a time, one per stream.  A target's sum is
// split over 16 roles of 16 streams: role w, stream s takes the sources
// (16 k + w) * 16 + s, k = 0, 1, ...; each stream adds its sources in order, a
// role's streams are added by exchange with stream ^ 15, ^ 7, ^ 2 and ^ 1, and
// the roles in order.  A workgroup's 16 waves are the roles, added through LDS.
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

// This wave's role for the 16 targets from t0 on, left in sum: sixteen sources
// at 16 w, 16 w + 256, ..., the next four rounds in flight.  na is a multiple
// of 64.
template <bool kRcp>
__device__ __forceinline__ void ds_block_role(const float2 *__restrict__ pos,
                                              const float *__restrict__ mass, uint32_t na,
                                              uint32_t t0, float eps2,
                                              float2 (&sum)[kDsRoles][kDsBlockTargets]) {
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t stream = lane & 15u, slot = lane >> 4;
    float tx[4], ty[4], ax[4], ay[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float2 p = pos[t0 + 4 * slot + r];
        tx[r] = p.x;
        ty[r] = p.y;
        ax[r] = 0.0f;
        ay[r] = 0.0f;
    }
    float ev = eps2;  // in a vector register: a scalar operand costs the second issue
    asm volatile("" : "+v"(ev));
    constexpr uint32_t kAhead = 4, kStep = 16 * kDsRoles;
    const uint32_t first = 16 * w + stream;
    DsSource q[kAhead];
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u)
        q[u] = ds_source(pos, mass, min(first + u * kStep, na - 16 + stream));
    for (uint32_t j = 16 * w; j < na; j += kAhead * kStep) {
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) {
            if (j + u * kStep >= na) break;
            const DsSource c = q[u];
            q[u] = ds_source(pos, mass, min(j + (u + kAhead) * kStep, na - 16) + stream);
            ds_add<kRcp>(c, tx, ty, ev, ax, ay);
        }
    }
    const float sx = ds_sum_streams(ax, lane), sy = ds_sum_streams(ay, lane);
    if ((lane & 3u) == 0) sum[w][4 * slot + (stream >> 2)] = make_float2(sx, sy);
}

// The roles' sums of target t, in order.
__device__ __forceinline__ float2 ds_block_sum(const float2 (&sum)[kDsRoles][kDsBlockTargets],
                                               uint32_t t) {
    float bx = 0.0f, by = 0.0f;
#pragma unroll
    for (uint32_t u = 0; u < kDsRoles; ++u) {
        bx = bx + sum[u][t].x;
        by = by + sum[u][t].y;
    }
    return make_float2(bx, by);
}

}  // namespace gsim
