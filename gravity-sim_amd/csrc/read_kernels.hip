// Readback: a system's particles in the caller's order.
//
// The Barnes-Hut state lives in the last step's sorted order.  Put back in
// order on the device, its three arrays leave as plain copies; in order on the
// host, 500,000 particles took 3.2 ms to read, of which the copies are 0.6.
// What bounds it now is the copy into the caller's pageable arrays.
//
// Up to kReadStageParticles the kernel writes straight into pinned host
// memory: one launch and one wait instead of a copy call for each array (5,000
// particles: direct sum 70 -> 22 us, Barnes-Hut 90 -> 33; the line is where the
// two meet).  The block takes 170 us to make, so a handle makes it for its
// second read.  Larger Barnes-Hut reads, us: 50,000 particles 150 -> 91, 500,000
// 3,197 -> 741, a million 6,810 -> 2,409.
#include "internal.hpp"

namespace gsim {
namespace {

// perm == nullptr: the state is in the caller's order.  stall: a counter that
// travels with the particles (the batch's radix sort), or nullptr.
__global__ __launch_bounds__(256) void read_kernel(
    const float2 *__restrict__ pos, const float2 *__restrict__ vel,
    const float *__restrict__ mass, const uint32_t *__restrict__ perm, uint32_t na, uint32_t n,
    float2 *__restrict__ pos_out, float2 *__restrict__ vel_out, float *__restrict__ mass_out,
    const uint32_t *__restrict__ stall, uint32_t *__restrict__ stall_out) {
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k == 0 && stall) *stall_out = *stall;
    if (k >= na) return;
    const uint32_t i = perm ? perm[k] : k;
    if (i >= n) return;  // padding
    pos_out[i] = pos[k];
    vel_out[i] = vel[k];
    mass_out[i] = mass[k];
}

}  // namespace

hipError_t read_launch(const float2 *pos, const float2 *vel, const float *mass,
                       const uint32_t *perm, uint32_t na, uint32_t n, const ReadTarget &out,
                       const uint32_t *stall, hipStream_t stream) {
    read_kernel<<<(na + 255) / 256, 256, 0, stream>>>(pos, vel, mass, perm, na, n, out.pos, out.vel,
                                                      out.mass, stall, out.stall);
    return hipGetLastError();
}

// The stage is one pinned block: positions, velocities, masses, the counter.
bool ReadStage::ready() {
    if (block) return true;
    if (!read_before) {
        read_before = true;
        return false;
    }
    if (hipHostMalloc(&block, kReadStageParticles * 20 + 64, hipHostMallocDefault) == hipSuccess)
        return true;
    (void)hipGetLastError();  // no pinned memory left: plain copies
    block = nullptr;
    return false;
}

void ReadStage::release() {
    if (block) (void)hipHostFree(block);
    block = nullptr;
}

ReadTarget ReadStage::target(size_t n) const {
    char *p = static_cast<char *>(block);
    return ReadTarget{reinterpret_cast<float2 *>(p), reinterpret_cast<float2 *>(p + 8 * n),
                      reinterpret_cast<float *>(p + 16 * n),
                      reinterpret_cast<uint32_t *>(p + 20 * kReadStageParticles)};
}

}  // namespace gsim
