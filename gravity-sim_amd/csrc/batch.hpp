// Batched multi-system stepping: many independent systems of uneven size in
// one device arena, all stepped by the same kernels (one launch per stage for
// every system), replayed from a hipGraph.  Sizes and membership live in
// device memory, so the captured graph stays valid while systems come and go
// within the arena's capacity.
#pragma once

#include <cstddef>
#include <map>
#include <vector>

#include "internal.hpp"

namespace gsim {

// One system's slot in the arena and its constants (host mirror + device copy).
struct SysDesc {
    uint32_t off, na, n, algo;       // arena offset (multiple of 64), padded/real count
    float eps2, theta2, kv, kp;      // softening^2, theta^2, velocity and position factors
    float dt, pad0;
    uint32_t bh_rank, sorted_base;   // Barnes-Hut: rank in the global sort, first sorted position
    uint32_t w;                      // Barnes-Hut vote width: 64 or 32
};

// Per Barnes-Hut rank, written by the emit kernel every step.
struct RankStats {
    uint32_t root;      // first node slot of the system's tree
    uint32_t end_slot;  // one past its last node slot
    uint32_t n_in;      // particles inside the domain
    uint32_t pad;
};

// The leaf kernel lists the (system, depth-5 tile) pairs holding leaves in
// kLiveLists lists picked by a hash of the pair, each with its own counter:
// one counter for all of them serialises thousands of same-address atomics.
constexpr uint32_t kLiveLists = 64;

// Workgroups of the direct-sum launch, and how many of them take blocks: one to
// a CU, so that the build beside it finds room, where the direct sums are a
// small part of the step; all, several to a CU, where they outlast the build.
// The line lies between seven mixes whose builds and walks differ in more than
// this ratio, so it is a fit, no model of which side takes longer: a mix near it
// may be on the slower side by some per cent.  Us a step beside / all, by direct-sum pairs per Barnes-Hut particle: 417 392 /
// 427, 450 236 / 255, 1,875 168 / 182, 2,000 447 / 439, 5,400 492 / 434, 27,000
// 472 / 406, no Barnes-Hut system 832 / 697.  256 beside: 128 +5%, 192 +1%, 512
// +6% at the mix above bb_ds_kernel.
constexpr uint32_t kBatchDsBlocks = 1024;
constexpr uint32_t kBatchDsBeside = 256;
constexpr uint64_t kBatchDsPairs = 1900;

// The walk launch's work list is dealt to kForceQueues interleaved queues
// (item i to queue i mod kForceQueues); the waves of queue q take its items
// one at a time from a counter, so a wave that drew light items takes more.
constexpr uint32_t kForceQueues = 64;
constexpr uint32_t kQueueStride = 32;  // words between their counters: a cache line each

struct BatchCounts {
    uint32_t n_bh;            // Barnes-Hut systems (ranks)
    uint32_t n_bh_particles;  // sum of their padded counts = sorted positions
    uint32_t n_items;         // work items, direct-sum blocks first
    uint32_t n_ds;            // direct-sum blocks
    uint32_t ds_groups;       // workgroups that take them (<= kBatchDsBlocks)
    uint32_t pad;
    uint32_t n_cells;         // cell nodes of all trees (emit)
    uint32_t n_leaves;        // occupied leaves of all trees (emit)
    uint32_t n_sys;           // all systems (direct sum and Barnes-Hut)
    uint32_t sort_stall;      // radix look-back waits that hit their bound since the
                              // membership was uploaded (never expected)
    uint32_t n_live[kLiveLists];  // (system, depth-5 tile) pairs holding leaves, per list
    unsigned long long accepts;  // Barnes-Hut real-lane acceptances, all steps
    unsigned long long visits;   // Barnes-Hut real-lane node visits, all steps
};
// the two totals are copied together
static_assert(offsetof(BatchCounts, visits) == offsetof(BatchCounts, accepts) + 8,
              "accepts and visits must be adjacent");

constexpr uint32_t kUnlimitedSteps = 0xffffffffu;

// Radix tiles of the batched sort: sort_rounds keys per thread (8, 12 or 16:
// tiles of 2,048, 3,072 or 4,096 keys; 12 by default, the autotuner picks).
// The look-back status words are sized for the smallest tile.  Each system is
// sorted by itself on its 21 bits of cell and killed bit, in three passes.
constexpr int kBatchSortRoundsDefault = 12;
constexpr int kBatchSortTileMin = 8 * kSortThreads;
constexpr uint32_t kBatchPasses = 3;

// Launch parameters of a batched step that never change results (the
// autotuner's knobs): persistent walk-launch width, radix tile size and the
// walk's issue-priority step and carry divisor (0: off).
struct BatchTune {
    // waves of the walk launch (four a SIMD are resident at once): 48 systems
    // of 1,030 to 63,279 particles 360 us a step with 4, 344 with 6, 346 with 8
    uint32_t waves_per_simd = 6;
    uint32_t sort_rounds = kBatchSortRoundsDefault;
    uint32_t run_queue = 64;   // <= kRunQueue (kept for the interface: the walk has no run queue)
    uint32_t prio_step = 32;   // summed chunks per priority level
    uint32_t prio_carry = 16;  // last step's chunks / this = the starting level
};

constexpr uint32_t kBatchRankShift = 21;                   // key = rank << 21 | cell (bit 20 = killed)
constexpr uint32_t kBatchMaxSystems = 1u << (32 - kBatchRankShift);  // 2048
constexpr uint32_t kBatchSentinel = 0xffffffffu;
constexpr uint32_t kMaxForceWaves = 1024u * 8u;  // persistent force launch: 8 waves per SIMD
// Largest arena: node slots (3 per particle) and offsets stay within
// 32-bit indices.
constexpr size_t kBatchMaxParticles = (0x7fffffffull / 8) / 64 * 64;

struct BatchDevice {
    // arena
    float2 *pos[2] = {}, *vel[2] = {};
    float *mass = nullptr;
    // membership
    SysDesc *desc = nullptr;
    uint32_t *bh_sys = nullptr, *bh_prefix = nullptr;  // [max_systems (+1)]
    uint2 *items = nullptr;
    uint32_t *remaining = nullptr;  // steps each system may still take (kUnlimitedSteps = no limit)
    BatchCounts *counts = nullptr;
    uint32_t *qnext = nullptr;  // [kForceQueues * kQueueStride] items drawn from each queue (zeroed each step)
    RankStats *stats = nullptr;
    // Barnes-Hut scratch over all sorted positions
    uint32_t *keys[2] = {}, *idx[2] = {};
    uint32_t *status = nullptr;       // [2][tile, group][tiles_cap * 256] radix look-back words, by pass parity
    uint32_t *digit_total = nullptr;  // [max_systems][kBatchPasses * 256] digit totals, zero between steps
    uint32_t *ichunk = nullptr;       // [item_capacity] chunks each work item summed last step (issue priority)
    uint32_t *block_cells = nullptr, *block_leaves = nullptr;
    int8_t *sdep = nullptr;
    uint32_t *cpos = nullptr, *sorted_src = nullptr;
    float4 *leaf_sum = nullptr;
    uint32_t *leaf_first = nullptr, *leaf_key = nullptr;
    uint32_t *tile_range = nullptr;
    uint32_t *live_tiles = nullptr;  // [kLiveLists][live_per_list] tiles with leaves, any order
    TileCell *top = nullptr;
    // nodes of all trees
    float4 *node4 = nullptr;
    uint4 *child = nullptr;           // a cell's children (kLeafMark)
    // each force wave's Barnes-Hut acceptances, then its node visits, in the
    // last step, summed into counts->accepts / visits by the step's last
    // kernel (a same-address atomic per wave costs more than the sum)
    unsigned long long *wave_acc = nullptr;  // [2 * kMaxForceWaves]
};

struct BatchSystem {
    gsim_params params;
    uint32_t off = 0, na = 0, n = 0;
    size_t node_reserve = 0;
    uint64_t steps = 0;          // steps taken (exact after a synchronisation)
    uint64_t added_at = 0;       // batch step count when the system joined
    uint64_t target = ~0ull;     // total steps to take (~0 = unlimited)
    bool spoilt = false;         // it stepped while the sort gave up: its state is invalid
};

}  // namespace gsim

struct gsim_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t side = nullptr;  // the direct sums, beside the build (captured with it)
    hipEvent_t fork = nullptr, join = nullptr;
    bool has_ds = false;         // the graphs hold the direct-sum launch
    bool wide = false;           // the graphs' walk addresses nodes by slot
    size_t narrow_nodes = gsim::kNarrowNodes;  // (tests lower it)
    size_t capacity = 0;        // particles (padded) in the arena
    size_t node_capacity = 0;   // node slots
    size_t partial_capacity = 0;  // direct-sum admission units
    size_t item_capacity = 0;
    uint32_t max_systems = 0;
    size_t tiles_cap = 0, blocks_cap = 0;
    // sort slots the graphs launch: what the members need, with room to grow
    // (not what the arena could hold: an idle slot is a workgroup that starts
    // and ends, three times a step); more drops the graphs
    uint32_t sort_slots = 256;
    gsim::BatchDevice d;
    std::map<uint32_t, gsim::BatchSystem> systems;  // id -> system
    std::map<uint32_t, uint32_t> free_ranges;       // arena offset -> length (units of particles)
    uint32_t next_id = 1;
    size_t nodes_reserved = 0, partial_used = 0;
    bool dirty = true;
    int cur = 0;
    hipGraphExec_t graph[2] = {nullptr, nullptr};
    gsim::BatchTune tune;
    gsim::ReadStage stage;
    uint64_t steps = 0;
    // host mirror of the membership arrays
    std::vector<gsim::SysDesc> h_desc;
    gsim::BatchCounts h_counts{};
};

namespace gsim {

hipError_t batch_launch_step(gsim_batch *b, int in, int out);

}  // namespace gsim
