// Batched stepping kernels: every kernel covers all systems of a batch and
// reads its sizes from device memory (BatchCounts), so a step captured once
// in a hipGraph serves any membership that fits the arena.
//
// Barnes-Hut systems are sorted each by itself, by cell, at consecutive sorted
// positions (keys rank << 21 | cell), and because node slots are position +
// scanned cell-node count, each system's pre-order tree lands
// contiguously in one global node array ([root, end_slot) per rank, recorded
// by the emit kernel).  The per-system semantics are those of the
// single-system kernels in bh_kernels.hip (same cells, same canonical order,
// same reduction association, same vote), so a system's result in a batch is
// bit-identical to its result alone.  Direct-sum systems run the roles of the
// single-system block kernel (ds_device.hpp), so they match bit for bit as
// well.
#include "batch.hpp"
#include "bh_device.hpp"
#include "ds_device.hpp"
#include "radix_device.hpp"

#include <algorithm>

namespace gsim {
namespace {

constexpr uint32_t kCellMask = (1u << 20) - 1u;
constexpr uint32_t kKilledBit = 1u << 20;

// ---- keys and sort -----------------------------------------------------------
// The particles come grouped by system (rank), so each system is sorted by
// itself, on the 21 bits of cell and killed bit alone: three passes instead of
// the four that keys with the rank in them take, digit totals per system, and
// look-back chains no longer than a system.  The radix tiles never cross a
// system: rank r's are the sort slots from bh_prefix[r] / tile keys + r on (at
// least as many as it needs), one workgroup a slot in launch order: the counter
// that dealt the tiles before was a chain of same-address atomics.
// Bound by latency.  48 systems of 1,000 to 64,000 particles: keys and sort
// 95 -> 45 us a step (a pass 19.4 -> 12.2), 12 systems up to 200,000: 101 -> 40
// (22.2 -> 10.9).

// The tile of a sort slot.
struct SortSeg {
    uint32_t r;              // rank
    uint32_t first, n;       // the system's sorted positions
    uint32_t slot0;          // its first slot
    uint32_t tile, tiles;    // this slot's tile of the system's tiles (tile >= tiles: none)
};

// Found by the whole workgroup (synchronises it): rank r's thread sees that
// the slot is r's.
__device__ __forceinline__ SortSeg sort_seg(const uint32_t *__restrict__ prefix, uint32_t nb,
                                            uint32_t slot, uint32_t tile_keys, SortSeg &sh) {
    if (threadIdx.x == 0) sh = SortSeg{0u, 0u, 0u, 0u, 0u, 0u};
    lds_barrier();
    for (uint32_t r = threadIdx.x; r < nb; r += kSortThreads) {
        const uint32_t f = prefix[r], e = prefix[r + 1];
        const uint32_t s0 = f / tile_keys + r, s1 = e / tile_keys + r + 1;
        if (slot >= s0 && (slot < s1 || r + 1 == nb))
            sh = SortSeg{r, f, e - f, s0, slot - s0, (e - f + tile_keys - 1) / tile_keys};
    }
    lds_barrier();
    return sh;
}

// Every particle's key (rank << 21 | cell; input of pass 0), the digit totals
// of its system's passes, and the step's clears.
template <int kR>
__global__ __launch_bounds__(kSortThreads) void bb_keys_kernel(
    const SysDesc *__restrict__ desc, const uint32_t *__restrict__ bh_sys,
    const uint32_t *__restrict__ bh_prefix, const uint32_t *__restrict__ remaining,
    BatchCounts *__restrict__ counts,
    float2 *__restrict__ pos, float *__restrict__ mass, float2 *__restrict__ pos_out,
    const float2 *__restrict__ vel, float2 *__restrict__ vel_out, uint32_t *__restrict__ keys,
    uint32_t *__restrict__ idx, uint32_t *__restrict__ tile_range,
    RankStats *__restrict__ stats, uint32_t *__restrict__ digit_total,
    uint32_t *__restrict__ status, size_t group_words) {
    __shared__ uint32_t h[kBatchPasses][256];
    __shared__ SortSeg seg_sh;
    constexpr uint32_t kTile = kR * kSortThreads;
    const uint32_t nb = counts->n_bh, th = threadIdx.x;
    const uint32_t tid = blockIdx.x * kSortThreads + th, stride = gridDim.x * kSortThreads;
    for (uint32_t t = tid; t < nb * kTileWords; t += stride) tile_range[t] = 0;
    for (uint32_t t = tid; t < nb; t += stride) stats[t] = RankStats{0u, 0u, 0u, 0u};
    for (uint32_t t = tid; t < kLiveLists; t += stride) counts->n_live[t] = 0;
    if (tid == 0) {
        counts->n_cells = 0;
        counts->n_leaves = 0;
    }
#pragma unroll
    for (uint32_t p = 0; p < kBatchPasses; ++p) h[p][th] = 0;
    const SortSeg seg = sort_seg(bh_prefix, nb, blockIdx.x, kTile, seg_sh);  // synchronises
    if (seg.tile >= seg.tiles) return;
    // the first radix pass's look-back words (each pass clears the next one's)
    status[(size_t)blockIdx.x * 256 + th] = 0;
    status[group_words + (size_t)blockIdx.x * 256 + th] = 0;
    const uint32_t di = bh_sys[seg.r], off = desc[di].off;
    const bool spent = remaining[di] == 0u;
    const uint32_t base = seg.tile * kTile + th, rank_bits = seg.r << kBatchRankShift;
    float2 p[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const uint32_t f = base + r * kSortThreads;
        p[r] = f < seg.n ? pos[off + f] : make_float2(0.0f, 0.0f);
    }
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const uint32_t f = base + r * kSortThreads;
        if (f >= seg.n) break;
        const uint32_t i = off + f;
        uint32_t c = kKilledBit;
        if (spent) {
            // Budget spent: the system keeps its state exactly (no kill of
            // particles that left the domain on its last step) and builds an
            // empty tree, so the force launch skips it.
            pos_out[i] = p[r];
            vel_out[i] = vel[i];
        } else {
            c = cell20(p[r].x, p[r].y);
            if (c == 0xffffffffu) {  // InitShader.comp:110-117
                const float k = -kSimSize * 2.0f;
                pos[i] = make_float2(k, k);
                pos_out[i] = make_float2(k, k);
                mass[i] = 0.0f;
                vel_out[i] = vel[i];
                c = kKilledBit;
            }
        }
        keys[seg.first + f] = rank_bits | c;
        idx[seg.first + f] = i;
        hist_add<kBatchPasses>(h, rank_bits | c);
    }
    lds_barrier();
    uint32_t *const total = digit_total + (size_t)seg.r * kBatchPasses * 256;
#pragma unroll
    for (uint32_t q = 0; q < kBatchPasses; ++q) {
        const uint32_t c = h[q][th];
        if (c) atomicAdd(&total[q * 256 + th], c);
    }
}

// Pass `pass` (digit (key >> 8 pass) & 255).  status: this pass's look-back
// words by slot, zeroed, the groups' group_words after the tiles' (a system's
// groups from its first slot on); status_next: the next pass's, zeroed here.
template <int kR>
__global__ __launch_bounds__(kSortThreads) void bb_onesweep_kernel(
    const uint32_t *__restrict__ keys_in, const uint32_t *__restrict__ idx_in,
    uint32_t *__restrict__ keys_out, uint32_t *__restrict__ idx_out,
    const uint32_t *__restrict__ bh_prefix, BatchCounts *__restrict__ counts, uint32_t pass,
    const uint32_t *__restrict__ digit_total, uint32_t *__restrict__ status,
    uint32_t *__restrict__ status_next, size_t group_words) {
    __shared__ SortShared<true, kR> sh;
    __shared__ SortSeg seg_sh;
    sort_tile_clear(sh);
    const SortSeg g = sort_seg(bh_prefix, counts->n_bh, blockIdx.x, kR * kSortThreads, seg_sh);
    if (g.tile >= g.tiles) return;
    status_next[(size_t)blockIdx.x * 256 + threadIdx.x] = 0;
    status_next[group_words + (size_t)blockIdx.x * 256 + threadIdx.x] = 0;
    uint32_t *const st = status + (size_t)g.slot0 * 256;
    sort_tile<true, kR>(keys_in + g.first, idx_in + g.first, keys_out + g.first, idx_out + g.first,
                        g.n, 8u * pass, g.tile, g.tiles, st, st + group_words,
                        digit_total + ((size_t)g.r * kBatchPasses + pass) * 256, 1u, 0u,
                        &counts->sort_stall, sh);
}

// ---- slot scan and emission ----------------------------------------------------

struct BPos {
    int sk, sk1;
    uint32_t ns, lf, rank, key;
    bool inside;
};

// s(k) and s(k+1) never cross a system boundary: the first position of a
// system behaves like position 0 of a single system, its last in-domain
// position like the last one.
__device__ __forceinline__ BPos bpos_info(const uint32_t *__restrict__ keys, uint32_t n,
                                          uint32_t k) {
    BPos q{-1, -1, 0u, 0u, 0u, 0u, false};
    if (k >= n) return q;
    q.key = keys[k];
    q.rank = q.key >> kBatchRankShift;
    if (q.key & kKilledBit) return q;
    q.inside = true;
    if (k > 0) {
        const uint32_t pk = keys[k - 1];
        if ((pk >> kBatchRankShift) == q.rank) q.sk = shared_depth(pk & kCellMask, q.key & kCellMask);
    }
    if (k + 1 < n) {
        const uint32_t nk = keys[k + 1];
        if ((nk >> kBatchRankShift) == q.rank && !(nk & kKilledBit))
            q.sk1 = shared_depth(q.key & kCellMask, nk & kCellMask);
    }
    q.ns = q.sk1 > q.sk ? (uint32_t)(q.sk1 - q.sk) : 0u;
    q.lf = q.sk < 10 ? 1u : 0u;
    return q;
}

__global__ __launch_bounds__(256) void bb_prep_kernel(const uint32_t *__restrict__ keys,
                                                      const BatchCounts *__restrict__ counts,
                                                      uint32_t *__restrict__ block_cells,
                                                      uint32_t *__restrict__ block_leaves,
                                                      uint32_t *__restrict__ digit_total) {
    __shared__ uint32_t wa[4], wb[4];
    const uint32_t n = counts->n_bh_particles;
    // the sort is done: its digit totals are cleared for the next step's
    const uint32_t words = counts->n_bh * kBatchPasses * 256;
    for (uint32_t t = blockIdx.x * 256 + threadIdx.x; t < words; t += gridDim.x * 256)
        digit_total[t] = 0;
    const uint32_t nblocks = (n + 255) / 256;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t blk = blockIdx.x; blk < nblocks; blk += gridDim.x) {
        const BPos q = bpos_info(keys, n, blk * 256 + threadIdx.x);
        uint32_t a = q.ns, b = q.lf;
        wave_scan2(a, b);
        if (lane == 63) {
            wa[wave] = a;
            wb[wave] = b;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            block_cells[blk] = wa[0] + wa[1] + wa[2] + wa[3];
            block_leaves[blk] = wb[0] + wb[1] + wb[2] + wb[3];
        }
        __syncthreads();
    }
}

// Exclusive scan of the per-block sums (blockIdx.x 0: cells, 1: leaves).
__global__ __launch_bounds__(1024) void bb_block_scan_kernel(uint32_t *__restrict__ a,
                                                             uint32_t *__restrict__ b,
                                                             const BatchCounts *__restrict__ counts) {
    __shared__ uint32_t wsum[16];
    scan_inplace_1024(blockIdx.x == 0 ? a : b, (counts->n_bh_particles + 255) / 256, wsum);
}

// Where a look-back of the sort gave up, its output is no permutation: every
// particle is taken as outside (no tree, no walk; bh_emit_kernel).
__global__ __launch_bounds__(256) void bb_emit_kernel(
    const uint32_t *__restrict__ keys, const uint32_t *__restrict__ sidx,
    const float2 *__restrict__ pos, const float *__restrict__ mass,
    BatchCounts *__restrict__ counts, const uint32_t *__restrict__ bh_prefix,
    const uint32_t *__restrict__ block_cells, const uint32_t *__restrict__ block_leaves,
    int8_t *__restrict__ sdep, uint32_t *__restrict__ cpos,
    uint32_t *__restrict__ leaf_first, uint32_t *__restrict__ leaf_key,
    float4 *__restrict__ node4, uint32_t *__restrict__ sorted_src,
    RankStats *__restrict__ stats) {
    __shared__ uint32_t wa[4], wb[4];
    const uint32_t n = counts->n_bh_particles;
    const uint32_t nblocks = (n + 255) / 256;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool stalled = counts->sort_stall != 0u;
    for (uint32_t blk = blockIdx.x; blk < nblocks; blk += gridDim.x) {
        const uint32_t k = blk * 256 + threadIdx.x;
        // the particle's gather does not depend on the scan below: start it first
        const uint32_t i = k < n && !stalled ? sidx[k] : 0u;
        const float2 p = k < n ? pos[i] : make_float2(0.0f, 0.0f);
        const float m = k < n ? mass[i] : 0.0f;
        BPos q = bpos_info(keys, n, k);
        if (stalled) q.inside = false;
        uint32_t a = q.ns, b = q.lf;
        wave_scan2(a, b);
        if (lane == 63) {
            wa[wave] = a;
            wb[wave] = b;
        }
        __syncthreads();
        uint32_t C = a - q.ns + block_cells[blk];
        uint32_t L = b - q.lf + block_leaves[blk];
        for (uint32_t w = 0; w < wave; ++w) {
            C += wa[w];
            L += wb[w];
        }
        __syncthreads();
        if (k >= n) continue;
        if (k + 1 == n && !stalled) {  // totals over all systems, and the end of the last leaf
            counts->n_cells = C + q.ns;
            counts->n_leaves = L + q.lf;
            leaf_first[L + q.lf] = q.inside ? k + 1 : n;
        }
        if (!q.inside) {
            sorted_src[k] = kBatchSentinel;
            continue;
        }
        const uint32_t slot = k + C + q.ns;
        node4[slot] = make_float4(p.x, p.y, m, 0.0f);
        sorted_src[k] = i;
        sdep[k] = (int8_t)q.sk;
        cpos[k] = C;
        if (q.lf) {
            leaf_first[L] = k;
            leaf_key[L] = q.key;
        }
        if (q.sk < 0) stats[q.rank].root = k + C;
        if (q.sk1 < 0) {
            stats[q.rank].end_slot = k + 1 + C + q.ns;
            stats[q.rank].n_in = k + 1 - bh_prefix[q.rank];
        }
    }
}

// ---- leaf sums ----------------------------------------------------------------

// The live list of (system r, depth-5 tile c), T = r kTiles + c: (c + 23 r)
// mod 64.  Each system gives each list exactly kTiles / 64 of its tiles, so a
// list never holds more than max_systems kTiles / 64 (its capacity), and the
// odd stride spreads the systems' few central tiles over the lists.
__device__ __forceinline__ uint32_t live_list(uint32_t T) {
    return ((T & (kTiles - 1u)) + 23u * (T / kTiles)) & (kLiveLists - 1u);
}

// Tile T's words in tile_range (kTileWords a system).
__device__ __forceinline__ uint32_t range_at(uint32_t T) {
    return T / kTiles * kTileWords + 2 * (T % kTiles);
}

__device__ __forceinline__ uint32_t tile_of(uint32_t key) {
    return (key >> kBatchRankShift) * kTiles + ((key >> 10) & (kTiles - 1));
}

// One leaf of system r: its record and, with two or more particles, its cell
// node, which comes right before its first particle's (node slot `first`).
__device__ __forceinline__ void bb_emit_leaf(const float4 &r, uint32_t L, uint32_t first,
                                             uint32_t n, float4 *__restrict__ leaf_sum,
                                             float4 *__restrict__ node4,
                                             uint4 *__restrict__ child) {
    leaf_sum[L] = make_float4(r.x, r.y, r.z, __uint_as_float(n));
    if (n >= 2u)
        emit_cell_at(TileCell{n, n + 1u, 0u, 0u, r.x, r.y, r.z, 0.0f}, (int)kTreeDepth, first - 1u,
                     make_uint4(n, 0u, 0u, kLeafMark), node4, child);
}

// The particles of leaf L, [f, e), and the node slot of the first: f + C(f + 1).
// The positions after a system's last in-domain one hold no C, but that one's
// C(f + 1) is what its tree ends with: end_slot - 1 - f.
struct LeafSpan {
    uint32_t f, e, first;
};

__device__ __forceinline__ LeafSpan leaf_span(uint32_t L, uint32_t key,
                                              const uint32_t *__restrict__ leaf_first,
                                              const uint32_t *__restrict__ bh_prefix,
                                              const RankStats *__restrict__ stats,
                                              const uint32_t *__restrict__ cpos) {
    const uint32_t r = key >> kBatchRankShift;
    const RankStats st = stats[r];
    const uint32_t sys_end = bh_prefix[r] + st.n_in;
    const uint32_t e = min(leaf_first[L + 1], sys_end);
    const uint32_t f = min(leaf_first[L], e);
    const uint32_t first = f + 1 < sys_end ? f + cpos[f + 1] : st.end_slot - 1u;
    return LeafSpan{f, e, first};
}

__global__ __launch_bounds__(256) void bb_leaf_kernel(
    const uint32_t *__restrict__ leaf_first, const uint32_t *__restrict__ leaf_key,
    const uint32_t *__restrict__ cpos, BatchCounts *counts,
    const uint32_t *__restrict__ bh_prefix, const RankStats *__restrict__ stats,
    float4 *__restrict__ leaf_sum, uint32_t *__restrict__ tile_range,
    uint32_t *__restrict__ live_tiles, uint32_t live_per_list, float4 *__restrict__ node4,
    uint4 *__restrict__ child) {
    __shared__ float4 stage[4][64];
    const uint32_t nl = counts->n_leaves;
    const uint32_t waves = gridDim.x * 4;
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t wave_id = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + w);
    // small leaves: each wave takes 64 consecutive leaves, one per lane
    for (uint32_t base = wave_id * 64; base < nl; base += waves * 64) {
        const uint32_t L = base + lane;
        if (L >= nl) continue;
        const uint32_t key = leaf_key[L];
        const LeafSpan p = leaf_span(L, key, leaf_first, bh_prefix, stats, cpos);
        if (p.e - p.f <= kSmallLeaf)
            bb_emit_leaf(lane_leaf_sum(node4, p.first, p.first + (p.e - p.f)), L, p.first,
                         p.e - p.f, leaf_sum, node4, child);
        const uint32_t T = tile_of(key);
        if (L == 0 || tile_of(leaf_key[L - 1]) != T) {
            tile_range[range_at(T)] = L;
            const uint32_t q = live_list(T);
            live_tiles[q * live_per_list + atomicAdd(&counts->n_live[q], 1u)] = T;
        }
        if (L + 1 == nl || tile_of(leaf_key[L + 1]) != T) tile_range[range_at(T) + 1] = L + 1;
    }
    // larger leaves: leaf L goes to wave L mod waves (neighbouring dense
    // leaves to different waves), streamed by the whole wave
    for (uint32_t i0 = 0; wave_id + i0 * waves < nl; i0 += 64) {
        const uint32_t L = wave_id + (i0 + lane) * waves;
        LeafSpan p{0u, 0u, 0u};
        if (L < nl) p = leaf_span(L, leaf_key[L], leaf_first, bh_prefix, stats, cpos);
        unsigned long long big = __ballot(L < nl && p.e - p.f > kSmallLeaf);
        while (big) {
            const uint32_t j = (uint32_t)__builtin_ctzll(big);
            big &= big - 1;
            const uint32_t n = __builtin_amdgcn_readfirstlane(__shfl(p.e - p.f, j, 64));
            const uint32_t first = __builtin_amdgcn_readfirstlane(__shfl(p.first, j, 64));
            const float4 r = wave_leaf_sum(stage[w], node4, first, first + n, lane);
            if (lane == 0)
                bb_emit_leaf(r, wave_id + (i0 + j) * waves, first, n, leaf_sum, node4, child);
        }
    }
}

// ---- dense reduction per (system, depth-5 tile), then per system --------------

// reduce_tile over the live lists; a system's last tile reduces its top.  One
// launch for what were two: 25.4 -> 16.6 us a step with 23 Barnes-Hut systems
// of up to 63,279 particles, 14.3 -> 10.0 with 12 of up to 104,223.
__global__ __launch_bounds__(256) void bb_tile_kernel(
    uint32_t *__restrict__ tile_range, const uint32_t *__restrict__ leaf_first,
    const uint32_t *__restrict__ leaf_key, const float4 *__restrict__ leaf_sum,
    const int8_t *__restrict__ sdep, const uint32_t *__restrict__ cpos,
    const BatchCounts *__restrict__ counts, const uint32_t *__restrict__ live_tiles,
    uint32_t live_per_list, float4 *__restrict__ node4, uint4 *__restrict__ child,
    TileCell *__restrict__ top) {
    __shared__ TileShared sh;
    // gridDim.x / kLiveLists workgroups per list (gridDim.x a multiple of kLiveLists)
    const uint32_t q = blockIdx.x % kLiveLists, per = gridDim.x / kLiveLists;
    const uint32_t nlive = counts->n_live[q];
    for (uint32_t i = blockIdx.x / kLiveLists; i < nlive; i += per) {  // only tiles holding leaves
        const uint32_t T = live_tiles[q * live_per_list + i], r = T / kTiles;
        reduce_tile(T % kTiles, tile_range + (size_t)r * kTileWords, leaf_first, leaf_key, leaf_sum,
                    nullptr, sdep, cpos, node4, child, top + (size_t)r * kTiles, kFixedR0, sh);
        lds_barrier();
    }
}

// ---- force: a launch for the direct sums, a persistent one for the walks --------

// Barnes-Hut group g of one system: the walk of bh_kernels.hip over the
// system's node range with its own constants, one wave per group.
template <int W, bool kWide>
__device__ void bb_walk_group(uint32_t g, const SysDesc &d, const RankStats &st, WalkShared &sh,
                              const uint32_t *__restrict__ sorted_src,
                              const float2 *__restrict__ pos, const float2 *__restrict__ vel,
                              const float4 *__restrict__ node4, const uint4 *__restrict__ child,
                              float2 *__restrict__ pos_out, float2 *__restrict__ vel_out,
                              uint32_t node_cap, unsigned long long &vis, unsigned long long &acc,
                              uint32_t *__restrict__ chunks_io, const BatchTune &tune) {
    constexpr int R = W / 8;
    constexpr uint32_t kLanes = 8 / R;  // lanes that end with a target
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t vsrc = sorted_src[d.sorted_base + g * W + (lane & (W - 1u))];
    const bool real = vsrc != kBatchSentinel;
    float2 vp = real ? pos[vsrc] : make_float2(0.0f, 0.0f);
    const unsigned long long rb = __ballot(real);
    const uint32_t nreal = (uint32_t)__popcll(W == 64 ? rb : rb & 0xffffffffull);
    // the killed sort last, so the group's first particle is real if any is
    vp.x = real ? vp.x : lane_value(vp.x, 0);
    vp.y = real ? vp.y : lane_value(vp.y, 0);
    const WalkTree tree{node4, child, uniform(st.root),
                        uniform(min(st.end_slot, node_cap)),
                        uniform(st.n_in)};
    // start at the issue priority this work item reached in the last step
    const uint32_t prio0 = tune.prio_carry ? *chunks_io / tune.prio_carry : 0u;
    float ax, ay;
    uint32_t chunks = 0;
    walk_group<W, R, kWide>(tree, sh, 0u, vp.x, vp.y, nreal, d.eps2, d.theta2, tune.prio_step,
                     prio0, ax, ay, vis, acc, chunks);
    if (lane == 0) *chunks_io = chunks;
    const uint32_t src = sorted_src[d.sorted_base + g * W + lane / kLanes];
    if (lane % kLanes != 0u || src == kBatchSentinel) return;
    const float2 p = pos[src], v = vel[src];
    const float nvx = v.x + ax * d.kv, nvy = v.y + ay * d.kv;
    pos_out[src] = make_float2(p.x + (v.x + nvx) * d.kp, p.y + (v.y + nvy) * d.kp);
    vel_out[src] = make_float2(nvx, nvy);
}

// The direct-sum systems' blocks of 16 targets (items [0, n_ds)), a workgroup a
// block: ds_block_kernel's additions in its order.  The blocks of one system
// follow each other, so that stepping by the grid spreads each system over all
// workgroups.  Bound by the VALU (alone 3.3e12 pairs a second).  One wave a
// block, role after role, inside the walks' launch took the time of the largest
// system's blocks: 25 systems of 1,030 to 6,128 particles alone 203 -> 123 us a
// step (the empty build's launches are 50 of each), with 23 Barnes-Hut systems
// 345 -> 311.
__global__ __launch_bounds__(64 * kDsRoles, 8) void bb_ds_kernel(
    const uint2 *__restrict__ items, const SysDesc *__restrict__ desc,
    const uint32_t *__restrict__ remaining, const BatchCounts *__restrict__ counts,
    const float2 *__restrict__ pos, const float2 *__restrict__ vel,
    const float *__restrict__ mass, float2 *__restrict__ pos_out, float2 *__restrict__ vel_out) {
    __shared__ float2 sum[kDsRoles][kDsBlockTargets];
    const uint32_t n = counts->n_ds, stride = counts->ds_groups;
    if (blockIdx.x >= stride) return;
    for (uint32_t it = blockIdx.x; it < n; it += stride) {
        const uint2 item = items[it];
        const SysDesc d = desc[item.x];
        const bool live = remaining[item.x] != 0u;
        const uint32_t t0 = item.y * kDsBlockTargets;
        const uint32_t i = d.off + t0 + (threadIdx.x & (kDsBlockTargets - 1u));
        const float2 p = pos[i], v = vel[i];
        if (live) ds_block_role<false>(pos + d.off, mass + d.off, d.na, t0, d.eps2, sum);
        lds_barrier();
        if (threadIdx.x < kDsBlockTargets) {
            float2 po = p, vo = v;  // budget spent: hold the state
            if (live) {
                const float2 b = ds_block_sum(sum, threadIdx.x);
                vo = make_float2(v.x + b.x * d.kv, v.y + b.y * d.kv);  // SimShader.comp:68-69
                po = make_float2(p.x + ((v.x + vo.x) * 0.5f) * d.dt,
                                 p.y + ((v.y + vo.y) * 0.5f) * d.dt);
            }
            pos_out[i] = po;
            vel_out[i] = vo;
        }
        lds_barrier();
    }
}

template <bool kWide>
__global__ __launch_bounds__(256) void bb_force_kernel(
    const uint2 *__restrict__ items, const SysDesc *__restrict__ desc,
    const uint32_t *__restrict__ remaining, const RankStats *__restrict__ stats,
    BatchCounts *__restrict__ counts,
    const uint32_t *__restrict__ sorted_src, const float2 *__restrict__ pos,
    const float2 *__restrict__ vel,
    const float4 *__restrict__ node4, const uint4 *__restrict__ child,
    float2 *__restrict__ pos_out, float2 *__restrict__ vel_out, uint32_t node_cap,
    unsigned long long *__restrict__ wave_acc, uint32_t *__restrict__ ichunk,
    uint32_t *__restrict__ qnext, BatchTune tune) {
    __shared__ WalkShared sh[4];
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t nitems = counts->n_items, n_ds = counts->n_ds;
    // this wave's queue (kForceQueues queues, each shared by the waves of one
    // residue): its first item goes by its place among them, the others are
    // drawn one at a time, the next one's ticket before the current item is
    // walked.  A wave without a first item draws none.  Two draws a wave from
    // counters side by side were a chain of 12,288 atomics on two cache lines:
    // the launch 140 -> 109 us with 9,600 items, 90 -> 54 with 1,300 to 5,200.
    const uint32_t wave = blockIdx.x * 4 + w, q = wave % kForceQueues;
    const uint32_t places = (gridDim.x * 4 + kForceQueues - 1 - q) / kForceQueues;
    uint32_t *const qctr = qnext + q * kQueueStride;
    auto draw = [&]() -> uint32_t {
        uint32_t j = 0;
        if (lane == 0) j = atomicAdd(qctr, 1u);
        return places + __builtin_amdgcn_readfirstlane(j);
    };
    unsigned long long acc = 0, vis = 0;
    uint32_t next = wave / kForceQueues;
    while (true) {
        const uint32_t it = n_ds + q + kForceQueues * next;
        if (it >= nitems) break;  // the queue is drained (every later ticket is beyond too)
        next = draw();
        const uint2 item = items[it];
        const SysDesc d = desc[item.x];
        const bool live = remaining[item.x] != 0u;
        const RankStats st = stats[d.bh_rank];
        // no particle inside the domain, or a spent budget (the keys
        // kernel has already written the system's output)
        if (!live || st.n_in == 0) continue;
        if (d.w == 32)
            bb_walk_group<32, kWide>(item.y, d, st, sh[w], sorted_src, pos, vel, node4, child,
                                     pos_out, vel_out, node_cap, vis, acc, &ichunk[it], tune);
        else
            bb_walk_group<64, kWide>(item.y, d, st, sh[w], sorted_src, pos, vel, node4, child,
                                     pos_out, vel_out, node_cap, vis, acc, &ichunk[it], tune);
    }
    if (lane == 0) {
        wave_acc[blockIdx.x * 4 + w] = acc;
        wave_acc[kMaxForceWaves + blockIdx.x * 4 + w] = vis;
    }
}

// End of a step: spend one step of every limited budget, and add the force
// waves' acceptances and visits to the running totals (one atomic each per
// block).
__global__ __launch_bounds__(256) void bb_finish_kernel(uint32_t *__restrict__ remaining,
                                                        BatchCounts *__restrict__ counts,
                                                        const unsigned long long *__restrict__ wave_acc,
                                                        uint32_t nwaves,
                                                        uint32_t *__restrict__ qnext) {
    __shared__ unsigned long long part[2][4];
    // the force launch's queue counters, for the next step
    if (blockIdx.x == 0 && threadIdx.x < kForceQueues) qnext[threadIdx.x * kQueueStride] = 0u;
    for (uint32_t s = blockIdx.x * 256 + threadIdx.x; s < counts->n_sys; s += gridDim.x * 256) {
        const uint32_t r = remaining[s];
        if (r != 0u && r != kUnlimitedSteps) remaining[s] = r - 1u;
    }
    unsigned long long a = 0, v = 0;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < nwaves; i += gridDim.x * 256) {
        a += wave_acc[i];
        v += wave_acc[kMaxForceWaves + i];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off, 64);
        v += __shfl_xor(v, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = a;
        part[1][threadIdx.x >> 6] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long ta = part[0][0] + part[0][1] + part[0][2] + part[0][3];
        const unsigned long long tv = part[1][0] + part[1][1] + part[1][2] + part[1][3];
        if (ta) atomicAdd(&counts->accepts, ta);
        if (tv) atomicAdd(&counts->visits, tv);
    }
}

}  // namespace

// One batched step: the direct sums on a stream beside the Barnes-Hut build of
// all BH systems, whose launches leave most of the GPU idle; then the walks.  Launched onto b->stream
// (captured into a graph by the caller).
hipError_t batch_launch_step(gsim_batch *b, int in, int out) {
    BatchDevice &d = b->d;
    hipStream_t st = b->stream;
    const uint32_t live_per_list = (uint32_t)(((size_t)b->max_systems * kTiles + kLiveLists - 1) / kLiveLists);
    if (b->has_ds) {
        hipError_t e = hipEventRecord(b->fork, st);
        if (e == hipSuccess) e = hipStreamWaitEvent(b->side, b->fork, 0);
        if (e != hipSuccess) return e;
        bb_ds_kernel<<<kBatchDsBlocks, 64 * kDsRoles, 0, b->side>>>(
            d.items, d.desc, d.remaining, d.counts, d.pos[in], d.vel[in], d.mass, d.pos[out],
            d.vel[out]);
        e = hipEventRecord(b->join, b->side);
        if (e != hipSuccess) return e;
    }
    const BatchTune &tune = b->tune;
    const uint32_t rounds = tune.sort_rounds;
    if (rounds != 8 && rounds != 12 && rounds != 16) return hipErrorInvalidValue;
    // passes: keys[0] -> keys[1] -> keys[0] -> keys[1]; look-back words
    // alternate between the two status halves (tile words, group words)
    const size_t group_words = 256 * b->tiles_cap, half = 2 * group_words;
#define GSIM_BB_SORT(R)                                                                          \
    do {                                                                                         \
        bb_keys_kernel<R><<<b->sort_slots, kSortThreads, 0, st>>>(                               \
            d.desc, d.bh_sys, d.bh_prefix, d.remaining, d.counts, d.pos[in], d.mass, d.pos[out], \
            d.vel[in], d.vel[out], d.keys[0], d.idx[0], d.tile_range, d.stats, d.digit_total,    \
            d.status, group_words);                                                              \
        for (uint32_t pass = 0; pass < kBatchPasses; ++pass) {                                   \
            const int i = pass & 1, o = i ^ 1;                                                   \
            bb_onesweep_kernel<R><<<b->sort_slots, kSortThreads, 0, st>>>(                       \
                d.keys[i], d.idx[i], d.keys[o], d.idx[o], d.bh_prefix, d.counts, pass,           \
                d.digit_total, d.status + half * i, d.status + half * o, group_words);           \
        }                                                                                        \
    } while (0)
    if (rounds == 8) GSIM_BB_SORT(8);
    else if (rounds == 12) GSIM_BB_SORT(12);
    else GSIM_BB_SORT(16);
#undef GSIM_BB_SORT
    const uint32_t *sk = d.keys[kBatchPasses & 1], *si = d.idx[kBatchPasses & 1];
    const uint32_t g_blk = (uint32_t)std::min<size_t>(b->blocks_cap, 4096);
    bb_prep_kernel<<<g_blk, 256, 0, st>>>(sk, d.counts, d.block_cells, d.block_leaves,
                                          d.digit_total);
    bb_block_scan_kernel<<<2, 1024, 0, st>>>(d.block_cells, d.block_leaves, d.counts);
    bb_emit_kernel<<<g_blk, 256, 0, st>>>(sk, si, d.pos[in], d.mass, d.counts, d.bh_prefix,
                                          d.block_cells, d.block_leaves, d.sdep, d.cpos,
                                          d.leaf_first, d.leaf_key, d.node4, d.sorted_src,
                                          d.stats);
    bb_leaf_kernel<<<4096, 256, 0, st>>>(d.leaf_first, d.leaf_key, d.cpos, d.counts, d.bh_prefix,
                                         d.stats, d.leaf_sum, d.tile_range, d.live_tiles,
                                         live_per_list, d.node4, d.child);
    const uint32_t g_tile = 4096;  // 64 workgroups per live list
    bb_tile_kernel<<<g_tile, 256, 0, st>>>(d.tile_range, d.leaf_first, d.leaf_key, d.leaf_sum,
                                           d.sdep, d.cpos, d.counts, d.live_tiles, live_per_list,
                                           d.node4, d.child, d.top);
    const uint32_t waves = 1024u * b->tune.waves_per_simd;
    auto *force = b->wide ? bb_force_kernel<true> : bb_force_kernel<false>;
    force<<<waves / 4, 256, 0, st>>>(d.items, d.desc, d.remaining, d.stats, d.counts, d.sorted_src,
                                               d.pos[in], d.vel[in], d.node4, d.child,
                                               d.pos[out], d.vel[out],
                                               (uint32_t)b->node_capacity, d.wave_acc, d.ichunk,
                                               d.qnext, tune);
    if (b->has_ds) {  // the finish counts the step as taken
        hipError_t e = hipStreamWaitEvent(st, b->join, 0);
        if (e != hipSuccess) return e;
    }
    bb_finish_kernel<<<8, 256, 0, st>>>(d.remaining, d.counts, d.wave_acc, waves, d.qnext);
    return hipGetLastError();
}

}  // namespace gsim
