// Barnes-Hut build and traversal for gfx950.
//
// Tree semantics follow the reference's fixed-domain quadtree
// (BarnesHutSimulation.cpp:885-918 and its seven shaders): domain [-500,500)^2,
// 1024^2 leaf grid, 11 levels, a node for every particle and for every cell
// holding >= 2 particles, flattened in pre-order with subtree sizes.  The
// build here is sparse instead of the reference's dense 1.4M-cell pyramid:
//
//   1. keys      20-bit Morton cell per particle (InitShader.comp:80-98); the
//                out-of-domain kill of InitShader.comp:110-117.
//   2. sort      stable LSD radix sort of (cell, index), 3 passes of 8 bits,
//                so a leaf's particles are in ascending index order: the
//                keys kernel counts the digits, then one launch per pass
//                (look-back).  Up to kSmallBuild particles steps 1 to 4 are
//                one launch of one workgroup.
//   3. prep      s(k) = depth shared by sorted keys k-1 and k; the cell nodes
//                that start at k are the depths in (s(k), s(k+1)], so an
//                exclusive scan C(k) of their number gives every pre-order
//                slot: particle k -> k + C(k+1); the depth-d cell starting at
//                k -> k + C(k) + (d - s(k) - 1).  Per-block counts here.
//   4. emit      the scan (each block adds up the counts before it), particle
//                nodes, sorted_src, leaf records.
//   5. leaf      leaf sums in ascending particle index (the canonical order of
//                the reference's float atomics, InitShader.comp:107-109) and
//                the leaf cells' nodes.
//   6. tile      one workgroup per depth-5 cell: the 32x32 leaf tile is
//                reduced in LDS level by level with ((c0+c1)+c2)+c3 exactly as
//                TreeInitShader.comp:78-83, counts y = sum + [sum > 1]; cells
//                with y > 1 are written as nodes (TreeMoveShader.comp:60-77),
//                with their children's subtree sizes.
//   7. top       the last tile workgroup to finish reduces the 1024 depth-5
//                cells to the root.
//   8. walk      groups of W sorted slots take the same cells; a node is
//                accepted iff all W particles accept it (ForceShader.comp:111-
//                141), then integrate (ForceShader.comp:145-150).
#include "bh_device.hpp"
#include "radix_device.hpp"

namespace gsim {
namespace {

// ---- 0. adaptive bounding box (opt-in; beyond the reference) -------------------
// Extremes of the finite positions: per-block partials, reduced by every
// workgroup of the keys kernel, which applies the box formula {cx, cy, h, r0}
// (order-independent, so exact).  One block's launch for it took 4.6 us (build
// with the box, 100,000 particles: 60.7 -> 59.1); up to kSmallBuild particles
// the one workgroup takes the extremes itself (1,000: 31.6 -> 27.2).

__device__ __forceinline__ void minmax4_wave(float &a, float &b, float &c, float &d) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a = fminf(a, __shfl_xor(a, off, 64));
        b = fmaxf(b, __shfl_xor(b, off, 64));
        c = fminf(c, __shfl_xor(c, off, 64));
        d = fmaxf(d, __shfl_xor(d, off, 64));
    }
}

__global__ __launch_bounds__(256) void bh_box_partial_kernel(const float2 *__restrict__ pos,
                                                             uint32_t na,
                                                             float4 *__restrict__ part) {
    __shared__ float4 wv[4];
    float x0 = __builtin_inff(), x1 = -__builtin_inff(), y0 = __builtin_inff(),
          y1 = -__builtin_inff();
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < na; i += gridDim.x * 256) {
        const float2 p = pos[i];
        if (!__builtin_isfinite(p.x) || !__builtin_isfinite(p.y)) continue;
        x0 = fminf(x0, p.x);
        x1 = fmaxf(x1, p.x);
        y0 = fminf(y0, p.y);
        y1 = fmaxf(y1, p.y);
    }
    minmax4_wave(x0, x1, y0, y1);
    if ((threadIdx.x & 63) == 0) wv[threadIdx.x >> 6] = make_float4(x0, x1, y0, y1);
    lds_barrier();
    if (threadIdx.x == 0) {
        float4 r = wv[0];
        for (int w = 1; w < 4; ++w) {
            r.x = fminf(r.x, wv[w].x);
            r.y = fmaxf(r.y, wv[w].y);
            r.z = fminf(r.z, wv[w].z);
            r.w = fmaxf(r.w, wv[w].w);
        }
        part[blockIdx.x] = r;
    }
}

// Centre, half edge and r0 of the box around extremes x0 <= x1, y0 <= y1.
__device__ __forceinline__ float4 box_of(float xmin, float xmax, float ymin, float ymax) {
    if (!(xmin <= xmax)) xmin = xmax = ymin = ymax = 0.0f;  // no finite particle
    const float cx = (xmin + xmax) * 0.5f, cy = (ymin + ymax) * 0.5f;
    const float w = fmaxf(xmax - xmin, ymax - ymin);
    float h = w * 0.501953125f;  // half the extent plus 2^-9: the farthest maps below 1024
    if (!(h >= 1e-3f)) h = 1e-3f;
    return make_float4(cx, cy, h, (h * h) * 2.0f);
}

// The box around every wave's extremes, in every thread of a workgroup of
// kWaves waves (synchronises it).
template <uint32_t kWaves>
__device__ __forceinline__ float4 box_of_group(float x0, float x1, float y0, float y1,
                                               float4 (&wv)[kWaves]) {
    minmax4_wave(x0, x1, y0, y1);
    if ((threadIdx.x & 63) == 0) wv[threadIdx.x >> 6] = make_float4(x0, x1, y0, y1);
    lds_barrier();
    float4 r = wv[0];
#pragma unroll
    for (uint32_t w = 1; w < kWaves; ++w) {
        const float4 o = wv[w];
        r = make_float4(fminf(r.x, o.x), fmaxf(r.y, o.y), fminf(r.z, o.z), fmaxf(r.w, o.w));
    }
    return box_of(r.x, r.y, r.z, r.w);
}

// ---- 1. keys ----------------------------------------------------------------

// kDeep: 30-bit keys of the 32768^2 grid (15-bit leaves) instead of 20-bit cells.
// One block of kR x kSortThreads particles (kR per thread) per workgroup.
// The digits of every radix pass are counted into digit_total, this build's
// half of the totals (kDigitCopies copies of 1024 words, workgroup b adding
// into copy b mod kDigitCopies; zeroed by the previous build's keys kernel,
// or at allocation), while digit_next, the other half, is zeroed for the next
// build; the radix passes' look-back words are zeroed as well.
// The particles are in the last step's sorted order: slot i holds the
// particle of original index perm[i].  Cells and slots are written at the
// original index (cells[perm[i]] = {cell, i}), so the sort runs over original
// indices, whose order breaks ties in a leaf, and carries each particle's
// slot.  An out-of-domain particle gets the killed key; its
// kill (InitShader.comp:110-117) is written by the emit kernel at the slot it
// sorts to.  kWalk: the last walk (write_next_key) and emit already wrote the
// cells; only the digits are counted.
template <bool kBox, bool kDeep, int kR, bool kWalk>
__global__ __launch_bounds__(kSortThreads) void bh_keys_kernel(
    const float2 *__restrict__ pos, const uint32_t *__restrict__ perm, uint32_t na,
    uint2 *__restrict__ cells, uint32_t *__restrict__ tile_range,
    uint32_t *__restrict__ digit_total, uint32_t *__restrict__ digit_next,
    uint32_t *__restrict__ status, uint32_t status_words, const float4 *__restrict__ box_part,
    uint32_t box_parts, float4 *__restrict__ box) {
    constexpr int kPasses = kDeep ? 4 : 3;
    __shared__ uint32_t h[kPasses][256];
    const uint32_t t = threadIdx.x;
    const uint32_t g = blockIdx.x * kSortThreads + t, stride = gridDim.x * kSortThreads;
    for (uint32_t j = g; j < kTileWords; j += stride) tile_range[j] = 0;
    for (uint32_t j = g; j < kDigitCopies * 1024; j += stride) digit_next[j] = 0;
    for (uint32_t j = g; j < status_words; j += stride) status[j] = 0;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) h[p][t] = 0;
    float4 bx = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if constexpr (kBox) {
        __shared__ float4 wv[kSortThreads / 64];
        const float inf = __builtin_inff();
        const float4 q = t < box_parts ? box_part[t] : make_float4(inf, -inf, inf, -inf);
        bx = box_of_group(q.x, q.y, q.z, q.w, wv);  // synchronises
        if (g == 0) *box = bx;
    } else {
        lds_barrier();
    }
    const uint32_t base = blockIdx.x * (kR * kSortThreads);
    if constexpr (kWalk) {
        uint32_t c[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            const uint32_t i = base + r * kSortThreads + t;
            c[r] = i < na ? cells[i].x : 0u;
        }
#pragma unroll
        for (int r = 0; r < kR; ++r)
            if (base + r * kSortThreads + t < na) hist_add<kPasses>(h, c[r]);
    } else {
    float2 pr[kR];
    uint32_t orig[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const uint32_t i = base + r * kSortThreads + t;
        pr[r] = i < na ? pos[i] : make_float2(0.0f, 0.0f);
        orig[r] = i < na ? perm[i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const uint32_t i = base + r * kSortThreads + t;
        if (i >= na) continue;
        const float2 p = pr[r];
        uint32_t c;
        if (kDeep) c = kBox ? cell30_box(p.x, p.y, bx.x, bx.y, bx.z) : cell30(p.x, p.y);
        else c = kBox ? cell20_box(p.x, p.y, bx.x, bx.y, bx.z) : cell20(p.x, p.y);
        if (c == 0xffffffffu) c = kDeep ? kKilledKeyDeep : kKilledKey;
        cells[orig[r]] = make_uint2(c, i);
        hist_add<kPasses>(h, c);
    }
    }
    lds_barrier();
    uint32_t *const copy = digit_total + (blockIdx.x % kDigitCopies) * 1024;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        const uint32_t n = h[p][t];
        if (n) atomicAdd(&copy[p * 256 + t], n);
    }
}

// ---- 2. stable LSD radix sort, one sweep per pass (radix_device.hpp) -----------

// One pass, one tile per workgroup: digit (key >> shift) & 255, with the
// two-level look-back (grouped_prefix).  digit_total: this pass's 256 totals,
// split over kDigitCopies copies 1024 words apart; status: this pass's
// [tiles][256] tile words followed by its [groups][256] group words, zeroed;
// Tiles of kR x kSortThreads keys.
template <int kR>
__global__ __launch_bounds__(kSortThreads) void radix_onesweep_kernel(
    const uint32_t *__restrict__ keys_in, const uint32_t *__restrict__ idx_in,
    const uint2 *__restrict__ cells_in, uint32_t *__restrict__ keys_out,
    uint32_t *__restrict__ idx_out, uint32_t n, uint32_t shift,
    const uint32_t *__restrict__ digit_total, uint32_t *__restrict__ status,
    uint32_t *__restrict__ stall) {
    __shared__ SortShared<false, kR> sh;
    sort_tile_clear(sh);  // the tile's first barrier follows its ranking
    // Tile = workgroup index: a tile only waits for lower ones, and every wait
    // ends (radix_device.hpp), also where a pass has more workgroups than fit
    // on the GPU at once (four a CU, from about 2,000,000 particles on).
    sort_tile<false, kR>(keys_in, idx_in, keys_out, idx_out, n, shift, blockIdx.x, gridDim.x,
                         status, status + (size_t)gridDim.x * 256, digit_total, kDigitCopies,
                         1024u, stall, sh, cells_in);
}

// ---- 3./4. slot scan and emission --------------------------------------------

// Per sorted position k: s(k), s(k+1) and the two scanned quantities.
struct PosInfo {
    int sk, sk1;
    uint32_t ns, lf;
    bool inside;
    uint32_t key;
    bool g10;  // first particle of an occupied depth-10 cell (15-bit leaves)
};

// bits: 10 (the reference's grid) or 15 (15-bit leaves); keys at or above
// 1 << 2*bits are killed particles.
__device__ __forceinline__ PosInfo pos_info(const uint32_t *__restrict__ keys, uint32_t na,
                                            uint32_t k, int bits) {
    PosInfo q{-1, -1, 0u, 0u, false, 0u, false};
    if (k >= na) return q;
    const uint32_t killed = 1u << (2 * bits);
    q.key = keys[k];
    if (q.key >= killed) return q;
    q.inside = true;
    q.sk = k == 0 ? -1 : shared_depth_bits(keys[k - 1], q.key, bits);
    if (k + 1 < na) {
        const uint32_t nk = keys[k + 1];
        if (nk < killed) q.sk1 = shared_depth_bits(q.key, nk, bits);
    }
    q.ns = q.sk1 > q.sk ? (uint32_t)(q.sk1 - q.sk) : 0u;
    q.lf = q.sk < bits ? 1u : 0u;
    q.g10 = q.sk < 10;
    return q;
}

// block_gran (15-bit leaves only, else nullptr): per-block counts of the
// occupied depth-10 cells as well.
__global__ __launch_bounds__(256) void bh_prep_kernel(const uint32_t *__restrict__ keys,
                                                      uint32_t na, int bits,
                                                      uint32_t *__restrict__ block_cells,
                                                      uint32_t *__restrict__ block_leaves,
                                                      uint32_t *__restrict__ block_gran) {
    __shared__ uint32_t wa[4], wb[4], wc[4];
    const PosInfo q = pos_info(keys, na, blockIdx.x * 256 + threadIdx.x, bits);
    uint32_t a = q.ns, b = q.lf;
    wave_scan2(a, b);
    const uint32_t c = (uint32_t)__popcll(__ballot(q.g10));
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 63) {
        wa[wave] = a;
        wb[wave] = b;
        wc[wave] = c;
    }
    lds_barrier();
    if (threadIdx.x == 0) {
        block_cells[blockIdx.x] = wa[0] + wa[1] + wa[2] + wa[3];
        block_leaves[blockIdx.x] = wb[0] + wb[1] + wb[2] + wb[3];
        if (block_gran) block_gran[blockIdx.x] = wc[0] + wc[1] + wc[2] + wc[3];
    }
}

// What the emission of a sorted position reads and writes.
struct EmitArgs {
    const float2 *pos, *vel;  // last step's order
    const float *mass;
    const uint32_t *perm_in;
    float2 *pos_out, *vel_out;
    float *mass_out;
    uint32_t *perm_out;
    uint2 *ncells;  // the next build's cells (nullptr: not kept)
    uint32_t na;
    int bits;
    int8_t *sdep;
    uint32_t *cpos, *leaf_first, *leaf_key;
    float4 *node4;
    uint32_t *sorted_src;
    BhCounters *ctr;
    uint32_t *gran_first, *gran_key;  // 15-bit leaves only, else nullptr
};

// Sorted position k: the particle of slot i in last step's order (p, m, the
// caller's index orig), with C cells, L leaves and G occupied depth-10 cells
// before it; k is its slot in the next order.
__device__ __forceinline__ void emit_position(const EmitArgs &e, const PosInfo &q, uint32_t k,
                                              uint32_t i, float2 p, float m, uint32_t orig,
                                              uint32_t C, uint32_t L, uint32_t G) {
    e.perm_out[k] = orig;
    if (!q.inside) {
        // killed (InitShader.comp:110-117): not walked; the reference leaves
        // vel_out stale, here it keeps the input velocity
        const float kk = -kSimSize * 2.0f;
        e.pos_out[k] = make_float2(kk, kk);
        e.vel_out[k] = e.vel[i];
        e.mass_out[k] = 0.0f;
        if (e.ncells)  // the next build's cell, where the walk writes the others
            e.ncells[orig] = make_uint2(e.bits == (int)kDeepBits ? kKilledKeyDeep : kKilledKey, k);
        e.sorted_src[k] = e.na;  // ClearShader.comp:81-82 sentinel
        if (k == 0) {            // nothing inside the domain
            e.ctr->n_in = 0;
            e.ctr->n_cells = 0;
            e.ctr->n_nodes = 0;
            e.ctr->n_leaves = 0;
            e.ctr->n_gran = 0;
            e.leaf_first[0] = 0;
            if (e.gran_first) e.gran_first[0] = 0;
        }
        return;
    }
    e.mass_out[k] = m;
    const uint32_t slot = k + C + q.ns;
    // ParticleSortShader.comp:99-107 (canonical order)
    e.node4[slot] = make_float4(p.x, p.y, m, 0.0f);
    e.sorted_src[k] = i;
    e.sdep[k] = (int8_t)q.sk;
    e.cpos[k] = C;
    if (q.lf) {
        e.leaf_first[L] = k;
        e.leaf_key[L] = q.key;
    }
    if (e.gran_first && q.g10) {
        e.gran_first[G] = k;
        e.gran_key[G] = q.key >> 10;  // the 20-bit cell
    }
    if (q.sk1 < 0) {  // last in-domain position
        e.ctr->n_in = k + 1;
        e.ctr->n_cells = C + q.ns;
        e.ctr->n_nodes = k + 1 + C + q.ns;
        e.ctr->n_leaves = L + q.lf;
        e.leaf_first[L + q.lf] = k + 1;
        e.ctr->n_gran = G + (q.g10 ? 1u : 0u);
        if (e.gran_first) e.gran_first[G + (q.g10 ? 1u : 0u)] = k + 1;
    }
}

// block_cells, block_leaves (and block_gran): bh_prep_kernel's per-block
// counts; each block adds up those of the blocks before it (integer sums, a
// few loads per thread) instead of a separate scan launch.  Where a look-back
// of the sort ever gave up (sort_stall), its output names slots that do not
// exist and has no order: every particle is taken as killed in place, so that
// nothing after this is out of bounds, and the handle's reads fail from then on.
__global__ __launch_bounds__(256) void bh_emit_kernel(
    const uint32_t *__restrict__ keys, const uint32_t *__restrict__ sidx, EmitArgs e,
    const uint32_t *__restrict__ block_cells, const uint32_t *__restrict__ block_leaves,
    const uint32_t *__restrict__ block_gran) {
    const uint32_t na = e.na;
    __shared__ uint32_t wa[4], wb[4], wc[4], pa[4], pb[4], pc[4];
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    // the particle now at sorted position k, from its slot i of the last
    // step's order (nearly the same order, so nearly sequential reads)
    const bool stalled = e.ctr->sort_stall != 0u;
    const uint32_t i = k >= na ? 0u : stalled ? k : sidx[k];
    const float2 p = k < na ? e.pos[i] : make_float2(0.0f, 0.0f);
    const float m = k < na ? e.mass[i] : 0.0f;
    const uint32_t orig = k < na ? e.perm_in[i] : 0u;
    // the counts of the blocks before this one, eight loads per thread at once
    uint32_t xa = 0, xb = 0, xc = 0;
    for (uint32_t j0 = threadIdx.x; j0 < blockIdx.x; j0 += 8 * 256) {
        uint32_t va[8], vb[8], vc[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            const uint32_t j = j0 + 256 * u;
            const bool in = j < blockIdx.x;
            va[u] = in ? block_cells[j] : 0u;
            vb[u] = in ? block_leaves[j] : 0u;
            vc[u] = in && block_gran ? block_gran[j] : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            xa += va[u];
            xb += vb[u];
            xc += vc[u];
        }
    }
    PosInfo q = pos_info(keys, na, k, e.bits);
    if (stalled) q.inside = false;
    uint32_t a = q.ns, b = q.lf;
    wave_scan2(a, b);
    const unsigned long long gb = __ballot(q.g10);
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        xa += __shfl_xor(xa, off, 64);
        xb += __shfl_xor(xb, off, 64);
        xc += __shfl_xor(xc, off, 64);
    }
    if (lane == 63) {
        wa[wave] = a;
        wb[wave] = b;
        wc[wave] = (uint32_t)__popcll(gb);
        pa[wave] = xa;
        pb[wave] = xb;
        pc[wave] = xc;
    }
    lds_barrier();
    uint32_t ea = a - q.ns + ((pa[0] + pa[1]) + (pa[2] + pa[3]));
    uint32_t eb = b - q.lf + ((pb[0] + pb[1]) + (pb[2] + pb[3]));
    uint32_t ec = (uint32_t)__popcll(gb & ((1ull << lane) - 1ull)) +
                  ((pc[0] + pc[1]) + (pc[2] + pc[3]));
    for (uint32_t w = 0; w < wave; ++w) {
        ea += wa[w];
        eb += wb[w];
        ec += wc[w];
    }
    if (k < na) emit_position(e, q, k, i, p, m, orig, ea, eb, ec);
}

// ---- 1.-4. in one workgroup: small builds ---------------------------------------

// Keys, sort, slot scan and emission of up to kSmallBuild particles by one
// workgroup of 16 waves.  Below that size each of the six launches it stands
// in for (keys, three sort passes, prep, emit) is bound by its own launch and
// its chain of loads; here the keys stay in LDS between the passes (digits of
// 7 bits, three passes; 15-bit leaves: 8 bits, four).  The limit is the LDS
// (64 KB of keys, indices and digit counts at 8,192 particles).
// It is bound by the vector units of its one CU (a ranking of 64 keys is 28
// operations) and, for the rest, by latency.  The whole build in us, six
// launches against this one: 64 particles 43 -> 20, 1,000 46 -> 24, 4,096
// 51 -> 33, 8,192 52 -> 45; 15-bit leaves and adaptive box 59 -> 37, 74 -> 50,
// 89 -> 65, 92 -> 85.
constexpr uint32_t kSmallBuild = 8192;
constexpr uint32_t kSmallWaves = 16;
constexpr uint32_t kSmallRows = kSmallBuild / (64 * kSmallWaves);  // keys per lane, at most

// A wave holds `rows` consecutive rows of 64 positions; cells and kWalk as in
// bh_keys_kernel, keys_out: the sorted keys.
template <bool kBox, bool kDeep, bool kWalk>
__global__ __launch_bounds__(64 * kSmallWaves) void bh_small_kernel(
    EmitArgs e, uint2 *__restrict__ cells, uint32_t *__restrict__ keys_out,
    uint32_t *__restrict__ tile_range, float4 *__restrict__ box) {
    constexpr uint32_t kBits = kDeep ? 8 : 7, kPasses = kDeep ? 4 : 3, kDigits = 1u << kBits;
    constexpr uint32_t kNone = 0xffffffffu;
    __shared__ uint32_t skey[kSmallBuild];
    __shared__ uint16_t sval[kSmallBuild];
    __shared__ uint32_t count[kSmallWaves * kDigits];
    __shared__ uint32_t wsum[kSmallWaves], wgran[kSmallWaves];
    const uint32_t na = e.na, t = threadIdx.x, lane = t & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t rows = (na + 64 * kSmallWaves - 1) / (64 * kSmallWaves);
    const uint32_t first = wave * rows * 64 + lane;  // row r: position first + 64 r
    for (uint32_t j = t; j < kTileWords; j += 64 * kSmallWaves) tile_range[j] = 0;
    uint32_t key[kSmallRows], val[kSmallRows], rank[kSmallRows];
    if constexpr (!kWalk) {
        float2 p[kSmallRows];
        uint32_t o[kSmallRows];
#pragma unroll
        for (uint32_t r = 0; r < kSmallRows; ++r) {
            const uint32_t k = first + 64 * r;
            if (r >= rows || k >= na) continue;
            p[r] = e.pos[k];
            o[r] = e.perm_in[k];
        }
        float4 bx = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if constexpr (kBox) {  // as bh_box_partial_kernel
            __shared__ float4 wv[kSmallWaves];
            float x0 = __builtin_inff(), x1 = -x0, y0 = x0, y1 = -x0;
#pragma unroll
            for (uint32_t r = 0; r < kSmallRows; ++r) {
                if (r >= rows || first + 64 * r >= na) continue;
                if (!__builtin_isfinite(p[r].x) || !__builtin_isfinite(p[r].y)) continue;
                x0 = fminf(x0, p[r].x);
                x1 = fmaxf(x1, p[r].x);
                y0 = fminf(y0, p[r].y);
                y1 = fmaxf(y1, p[r].y);
            }
            bx = box_of_group(x0, x1, y0, y1, wv);
            if (t == 0) *box = bx;
        }
#pragma unroll
        for (uint32_t r = 0; r < kSmallRows; ++r) {
            const uint32_t k = first + 64 * r;
            if (r >= rows || k >= na) continue;
            const float x = p[r].x, y = p[r].y;
            uint32_t c;
            if (kDeep) c = kBox ? cell30_box(x, y, bx.x, bx.y, bx.z) : cell30(x, y);
            else c = kBox ? cell20_box(x, y, bx.x, bx.y, bx.z) : cell20(x, y);
            if (c == kNone) c = kDeep ? kKilledKeyDeep : kKilledKey;
            cells[o[r]] = make_uint2(c, k);
            skey[o[r]] = c;
            sval[o[r]] = (uint16_t)k;
        }
        lds_barrier();
    }
#pragma unroll
    for (uint32_t r = 0; r < kSmallRows; ++r) {
        const uint32_t k = first + 64 * r;
        key[r] = kNone;
        val[r] = 0;
        if (r < rows && k < na) {
            if (kWalk) {
                const uint2 kv = cells[k];
                key[r] = kv.x;
                val[r] = kv.y;
            } else {
                key[r] = skey[k];
                val[r] = sval[k];
            }
        }
    }
    uint32_t *const mine = count + wave * kDigits;
#pragma unroll 1
    for (uint32_t pass = 0; pass < kPasses; ++pass) {
        const uint32_t shift = pass * kBits;
#pragma unroll
        for (uint32_t d = 0; d < kDigits; d += 64) mine[d + lane] = 0;
        wave_lds_order();
        // ranks within the wave, a row after the other
#pragma unroll
        for (uint32_t r = 0; r < kSmallRows; ++r) {
            if (r >= rows) break;
            const bool valid = key[r] != kNone;
            const uint32_t d = (key[r] >> shift) & (kDigits - 1);
            const uint64_t m = digit_peers<(int)kBits>(d, valid);
            const uint32_t before = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            const uint32_t n = mine[d];
            rank[r] = n + before;
            wave_lds_order();
            if (valid && before == 0) mine[d] = n + (uint32_t)__popcll(m);
            wave_lds_order();
        }
        lds_barrier();
        // digit t: where each wave's keys of it go
        uint32_t n[kSmallWaves], sum = 0, unused = 0;
        if (t < kDigits) {
#pragma unroll
            for (uint32_t w = 0; w < kSmallWaves; ++w) n[w] = count[w * kDigits + t];
#pragma unroll
            for (uint32_t w = 0; w < kSmallWaves; ++w) sum += n[w];
        }
        uint32_t at = sum;
        if (t < kDigits) {
            wave_scan2(at, unused);
            if (lane == 63) wsum[wave] = at;
        }
        lds_barrier();
        if (t < kDigits) {
            at -= sum;
            for (uint32_t w = 0; w < wave; ++w) at += wsum[w];
#pragma unroll
            for (uint32_t w = 0; w < kSmallWaves; ++w) {
                count[w * kDigits + t] = at;
                at += n[w];
            }
        }
        lds_barrier();
#pragma unroll
        for (uint32_t r = 0; r < kSmallRows; ++r) {
            if (r >= rows || key[r] == kNone) continue;
            const uint32_t to = mine[(key[r] >> shift) & (kDigits - 1)] + rank[r];
            skey[to] = key[r];
            sval[to] = (uint16_t)val[r];
        }
        lds_barrier();
#pragma unroll
        for (uint32_t r = 0; r < kSmallRows; ++r) {
            const uint32_t k = first + 64 * r;
            if (r >= rows || k >= na) continue;
            key[r] = skey[k];
            val[r] = sval[k];
        }
    }
    // the particles of the sorted positions, all loads ahead of the scan
    float2 p[kSmallRows];
    float m[kSmallRows];
    uint32_t orig[kSmallRows];
#pragma unroll
    for (uint32_t r = 0; r < kSmallRows; ++r) {
        if (r >= rows || key[r] == kNone) continue;
        p[r] = e.pos[val[r]];
        m[r] = e.mass[val[r]];
        orig[r] = e.perm_in[val[r]];
    }
    // cells and leaves before each position: cells in the low 18 bits (at most
    // 16 a particle), leaves above (at most one)
    uint32_t ahead[kSmallRows], gahead[kSmallRows], run = 0, grun = 0;
#pragma unroll
    for (uint32_t r = 0; r < kSmallRows; ++r) {
        if (r >= rows) break;
        const PosInfo q = pos_info(skey, na, first + 64 * r, e.bits);
        const uint32_t own = q.ns | q.lf << 18;
        uint32_t incl = own, unused = 0;
        wave_scan2(incl, unused);
        ahead[r] = run + incl - own;
        run += __builtin_amdgcn_readlane(incl, 63);
        const unsigned long long g = __ballot(q.g10);
        gahead[r] = grun + (uint32_t)__popcll(g & ((1ull << lane) - 1ull));
        grun += (uint32_t)__popcll(g);
    }
    if (lane == 0) {
        wsum[wave] = run;
        wgran[wave] = grun;
    }
    lds_barrier();
    uint32_t base = 0, gbase = 0;
    for (uint32_t w = 0; w < wave; ++w) {
        base += wsum[w];
        gbase += wgran[w];
    }
#pragma unroll
    for (uint32_t r = 0; r < kSmallRows; ++r) {
        const uint32_t k = first + 64 * r;
        if (r >= rows || k >= na) continue;
        const uint32_t a = base + ahead[r];
        const PosInfo q = pos_info(skey, na, k, e.bits);
        keys_out[k] = key[r];
        emit_position(e, q, k, val[r], p[r], m[r], orig[r], a & 0x3ffffu, a >> 18,
                      gbase + gahead[r]);
    }
}

// ---- 5. leaf sums --------------------------------------------------------------

constexpr uint32_t kLeafBlocks = 4096;
constexpr uint32_t kBoxParts = 256;  // blocks of the box reduction

// The node slot of the particle at sorted position f: f + C(f + 1).
__device__ __forceinline__ uint32_t particle_slot(uint32_t f, uint32_t n_in, uint32_t n_cells,
                                                  const uint32_t *__restrict__ cpos) {
    return f + (f + 1 < n_in ? cpos[f + 1] : n_cells);
}

// A leaf's record: its sums to leaf_sum (15-bit leaves: to nsum at its cell
// node, for the level reduction) and, with two or more particles, its cell
// node, which comes right before its first particle's.
__device__ __forceinline__ void emit_leaf(const float4 &r, uint32_t L, uint32_t first,
                                          uint32_t n, int bits, float4 *__restrict__ leaf_sum,
                                          float4 *__restrict__ node4,
                                          uint4 *__restrict__ child, float4 *__restrict__ nsum,
                                          float r0) {
    const float4 sum = make_float4(r.x, r.y, r.z, __uint_as_float(n));
    if (!nsum) leaf_sum[L] = sum;
    if (n < 2u) return;
    emit_cell_at(TileCell{n, n + 1u, 0u, 0u, r.x, r.y, r.z, 0.0f}, bits, first - 1u,
                 make_uint4(n, 0u, 0u, kLeafMark), node4, child, r0);
    if (nsum) nsum[first - 1u] = sum;
}

// The sum runs over the leaf's particles in sorted (= ascending index) order,
// the canonical order of the reference's float atomics: small leaves one per
// lane, larger ones one per wave (wave_leaf_sum).  nsum != nullptr: 15-bit
// leaves, which have no tiles.
__global__ __launch_bounds__(256) void bh_leaf_kernel(
    const uint32_t *__restrict__ leaf_first, const uint32_t *__restrict__ leaf_key,
    const uint32_t *__restrict__ cpos, const BhCounters *__restrict__ ctr, int bits,
    float4 *__restrict__ leaf_sum, uint32_t *__restrict__ tile_range,
    float4 *__restrict__ node4, uint4 *__restrict__ child, float4 *__restrict__ nsum,
    const float *__restrict__ box) {
    __shared__ float4 stage[4][64];
    const uint32_t n_in = ctr->n_in, nl = ctr->n_leaves, ncells = ctr->n_cells;
    const bool deep = nsum != nullptr;
    const float r0 = box ? box[3] : kFixedR0;
    const uint32_t waves = gridDim.x * 4;
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t wave_id = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + w);
    // larger leaves: leaf L goes to wave (waves - 1 - L) mod waves, so the
    // largest ones (dense cores, low L when few) avoid the first waves, which
    // hold the small leaves; neighbouring dense leaves go to different waves;
    // each is streamed by the whole wave
    const uint32_t rw = waves - 1u - wave_id;
    for (uint32_t i0 = 0; rw + i0 * waves < nl; i0 += 64) {
        const uint32_t L = rw + (i0 + lane) * waves;
        uint32_t f = 0, e = 0;
        if (L < nl) {
            e = min(leaf_first[L + 1], n_in);
            f = min(leaf_first[L], e);
        }
        unsigned long long big = __ballot(L < nl && e - f > kSmallLeaf);
        while (big) {
            const uint32_t j = (uint32_t)__builtin_ctzll(big);
            big &= big - 1;
            const uint32_t bf = __builtin_amdgcn_readfirstlane(__shfl(f, j, 64));
            const uint32_t be = __builtin_amdgcn_readfirstlane(__shfl(e, j, 64));
            const uint32_t first = particle_slot(bf, n_in, ncells, cpos);
            const float4 r = wave_leaf_sum(stage[w], node4, first, first + (be - bf), lane);
            if (lane == 0)
                emit_leaf(r, rw + (i0 + j) * waves, first, be - bf, bits, leaf_sum, node4, child,
                          nsum, r0);
        }
    }
    // small leaves: each wave takes 64 consecutive leaves, one per lane
    for (uint32_t base = wave_id * 64; base < nl; base += waves * 64) {
        const uint32_t L = base + lane;
        if (L >= nl) continue;
        const uint32_t e = min(leaf_first[L + 1], n_in);
        const uint32_t f = min(leaf_first[L], e);
        if (e - f <= kSmallLeaf) {
            const uint32_t first = particle_slot(f, n_in, ncells, cpos);
            emit_leaf(lane_leaf_sum(node4, first, first + (e - f)), L, first, e - f, bits,
                      leaf_sum, node4, child, nsum, r0);
        }
        if (!deep) {
            const uint32_t T = leaf_key[L] >> 10;
            if (L == 0 || (leaf_key[L - 1] >> 10) != T) {
                tile_range[2 * T] = L;
            }
            if (L + 1 == nl || (leaf_key[L + 1] >> 10) != T) tile_range[2 * T + 1] = L + 1;
        }
    }
}

// ---- 6'. sparse level reduction (15-bit leaves) ---------------------------------

// The sums of the depth-d cell (>= 2 particles) that starts at sorted position
// k, from its children in pre-order at slot + 1 on: a particle node contributes
// 0 + m*p, a cell node its sums in nsum; each child's quadrant comes from the
// key bits of its first particle.  Sums are ((c0 + c1) + c2) + c3 with an
// empty quadrant +0: the dense tile reduction's rule, evaluated only where
// particles are.  Returns (sx, sy, sm), the particle count n, the subtree size
// y and the children's sizes by quadrant.
struct CellSums {
    TileCell c;
    uint4 sizes;
};

__device__ __forceinline__ uint32_t subtree_size(uint4 ch) {
    return ch.w == kLeafMark ? ch.x + 1u : ch.x + ch.y + ch.z + ch.w + 1u;
}

__device__ __forceinline__ CellSums child_sums(const uint32_t *__restrict__ keys,
                                               const float4 *__restrict__ node4,
                                               const uint4 *__restrict__ child,
                                               const float4 *__restrict__ nsum, uint32_t k,
                                               uint32_t slot, int d, uint32_t n_in,
                                               uint32_t n_nodes) {
    const uint32_t shift = 2u * (kDeepBits - 1u - (uint32_t)d);  // child quadrant bits
    const uint32_t prefix = keys[k] >> (shift + 2u);
    float4 v0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), v1 = v0, v2 = v0, v3 = v0;
    uint4 sizes = make_uint4(0u, 0u, 0u, 0u);
    uint32_t c = slot + 1u, f = k, n = 0u, y = 1u;
    // at most four children (distinct quadrants)
    for (int it = 0; it < 4 && f < n_in && c < n_nodes; ++it) {
        // one round of loads per child: everything a cell or a particle needs
        // is read before the record says which one the child is
        const uint32_t key = keys[f];
        const float4 p = node4[c];
        const uint4 ch = child[c];
        const float4 s = nsum[c];
        if ((key >> (shift + 2u)) != prefix) break;
        float4 v;
        uint32_t cn = 1u, cy = 1u;
        if (p.w <= 0.0f) {  // a particle node: pos *= mass, InitShader.comp:102
            v = make_float4(0.0f + p.x * p.z, 0.0f + p.y * p.z, 0.0f + p.z, 0.0f);
        } else {
            v = s;
            cn = __float_as_uint(v.w);
            cy = subtree_size(ch);
        }
        const uint32_t q = (key >> shift) & 3u;
        if (q == 0u) { v0 = v; sizes.x = cy; }
        else if (q == 1u) { v1 = v; sizes.y = cy; }
        else if (q == 2u) { v2 = v; sizes.z = cy; }
        else { v3 = v; sizes.w = cy; }
        n += cn;
        y += cy;
        f += cn;
        c += cy;
    }
    return CellSums{TileCell{n, y, k, 0u, ((v0.x + v1.x) + v2.x) + v3.x,
                             ((v0.y + v1.y) + v2.y) + v3.y, ((v0.z + v1.z) + v2.z) + v3.z, 0.0f},
                    sizes};
}

// One launch per depth d = 14..11: every cell node of depth d (a sorted
// position k with s(k) < d <= s(k+1) starts one) gets its node and its sums.
__global__ __launch_bounds__(256) void bh_level_kernel(
    const uint32_t *__restrict__ keys, const int8_t *__restrict__ sdep,
    const uint32_t *__restrict__ cpos, const BhCounters *__restrict__ ctr,
    float4 *__restrict__ node4, uint4 *__restrict__ child, float4 *__restrict__ nsum, int d,
    const float *__restrict__ box) {
    const uint32_t n_in = ctr->n_in, n_nodes = ctr->n_nodes;
    const float r0 = box ? box[3] : kFixedR0;
    for (uint32_t k = blockIdx.x * 256 + threadIdx.x; k < n_in; k += gridDim.x * 256) {
        const int sk = sdep[k];
        const int sk1 = k + 1 < n_in ? (int)sdep[k + 1] : -1;
        if (!(sk < d && d <= sk1)) continue;
        const uint32_t slot = k + cpos[k] + (uint32_t)(d - sk - 1);
        const CellSums r = child_sums(keys, node4, child, nsum, k, slot, d, n_in, n_nodes);
        emit_cell_at(r.c, d, slot, r.sizes, node4, child, r0);
        nsum[slot] = make_float4(r.c.sx, r.c.sy, r.c.sm, __uint_as_float(r.c.n));
    }
}

// Depth 10 and up with 15-bit leaves: the cells of depth <= 10 are those of a
// 10-bit tree over the same particles, so the dense tile and top kernels
// reduce them once each occupied depth-10 cell (granule) has its record: the
// sums of its depth-10 cell (child_sums; its node is written here) when it
// holds >= 2 particles, else 0 + m*p of its one particle; particle count;
// subtree size.  Also marks each depth-5 tile's granule range for the tile
// kernel.
__global__ __launch_bounds__(256) void bh_gran_kernel(
    const uint32_t *__restrict__ keys, const int8_t *__restrict__ sdep,
    const uint32_t *__restrict__ cpos, const BhCounters *__restrict__ ctr,
    float4 *__restrict__ node4, uint4 *__restrict__ child,
    const float4 *__restrict__ nsum, const uint32_t *__restrict__ gran_first,
    const uint32_t *__restrict__ gran_key, float4 *__restrict__ gran_sum,
    uint32_t *__restrict__ gran_y, uint32_t *__restrict__ tile_range,
    const float *__restrict__ box) {
    const uint32_t n_in = ctr->n_in, n_nodes = ctr->n_nodes, ng = ctr->n_gran;
    const float r0 = box ? box[3] : kFixedR0;
    for (uint32_t L = blockIdx.x * 256 + threadIdx.x; L < ng; L += gridDim.x * 256) {
        const uint32_t k = gran_first[L];
        const int sk = sdep[k];
        const int sk1 = k + 1 < n_in ? (int)sdep[k + 1] : -1;
        if (sk1 >= 10) {
            const uint32_t slot = k + cpos[k] + (uint32_t)(10 - sk - 1);
            const CellSums r = child_sums(keys, node4, child, nsum, k, slot, 10, n_in, n_nodes);
            emit_cell_at(r.c, 10, slot, r.sizes, node4, child, r0);
            gran_sum[L] = make_float4(r.c.sx, r.c.sy, r.c.sm, __uint_as_float(r.c.n));
            gran_y[L] = r.c.y;
        } else {
            const float4 p = node4[particle_slot(k, n_in, ctr->n_cells, cpos)];
            gran_sum[L] = make_float4(0.0f + p.x * p.z, 0.0f + p.y * p.z, 0.0f + p.z,
                                      __uint_as_float(1u));
            gran_y[L] = 1u;
        }
        const uint32_t T = gran_key[L] >> 10;
        if (L == 0 || (gran_key[L - 1] >> 10) != T) {
            tile_range[2 * T] = L;
        }
        if (L + 1 == ng || (gran_key[L + 1] >> 10) != T) tile_range[2 * T + 1] = L + 1;
    }
}

// ---- 6./7. dense reduction per tile, then the top ------------------------------

__global__ __launch_bounds__(256) void bh_tile_kernel(
    uint32_t *__restrict__ tile_range, const uint32_t *__restrict__ leaf_first,
    const uint32_t *__restrict__ leaf_key, const float4 *__restrict__ leaf_sum,
    const int8_t *__restrict__ sdep, const uint32_t *__restrict__ cpos,
    float4 *__restrict__ node4, uint4 *__restrict__ child, TileCell *__restrict__ top,
    const float *__restrict__ box, const uint32_t *__restrict__ leaf_y) {
    __shared__ TileShared sh;
    const uint32_t T = blockIdx.x;
    if (tile_range[2 * T] == tile_range[2 * T + 1]) return;  // the whole workgroup: empty
    reduce_tile(T, tile_range, leaf_first, leaf_key, leaf_sum, leaf_y, sdep, cpos, node4, child,
                top, box ? box[3] : kFixedR0, sh);
}

// ---- 8. traversal + integrate ----------------------------------------------------

// The next build's sort input, written by the walk on the fixed domain: the
// cell of the particle's new position (InitShader.comp:73-119), at the
// particle's caller index o = perm[slot] (cells[o] = {cell, slot}), so the
// next build reads cells instead of positions.  cells == nullptr: the next
// build computes the cells itself (adaptive box, first step).
struct NextKeys {
    const uint32_t *perm;  // this step's output order: slot -> caller's index
    uint2 *cells;
    uint32_t deep;  // 30-bit cells
};

__device__ __forceinline__ void write_next_key(const NextKeys &nk, uint32_t slot, float2 p) {
    uint32_t c = nk.deep ? cell30(p.x, p.y) : cell20(p.x, p.y);
    if (c == 0xffffffffu) c = nk.deep ? kKilledKeyDeep : kKilledKey;
    nk.cells[nk.perm[slot]] = make_uint2(c, slot);
}

// The walk's launch order, by workgroup (four consecutive groups, the launch
// unit): by last step's walk cost (the four groups' real-lane visits, gvis),
// heaviest first, in buckets of a quarter of the mean (the last bucket holds
// everything from 7.75x the mean up) and by index within a bucket, so the
// dense-core groups start in the launch's first round and the light ones
// fill its end.  No costs yet (first step): index order.  Which wave walks a
// group never changes a result.  One workgroup: it is bound by its own
// instruction count, which ordering units of four groups keeps small.
constexpr uint32_t kOrderBuckets = 32;
constexpr uint32_t kOrderAhead = 4;

// The lanes of the wave whose 5-bit bucket equals this lane's (five ballots,
// whatever the number of distinct buckets); q = kOrderBuckets: no unit.
__device__ __forceinline__ unsigned long long bucket_peers(uint32_t q) {
    unsigned long long m = __ballot(q < kOrderBuckets);
#pragma unroll
    for (int bit = 0; bit < 5; ++bit) {
        const unsigned long long b = __ballot((q >> bit) & 1u);
        m &= ((q >> bit) & 1u) ? b : ~b;
    }
    return m;
}

__global__ __launch_bounds__(1024) void bh_order_plan_kernel(
    const unsigned long long *__restrict__ gvis, uint32_t groups, uint32_t *__restrict__ order) {
    __shared__ unsigned long long wsum[16];
    __shared__ uint32_t base[2][kOrderBuckets];
    __shared__ uint32_t wcnt[2][16][kOrderBuckets];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint32_t units = (groups + 3) / 4;
    const unsigned long long below = (1ull << lane) - 1ull;
    // a unit's cost, clamped to 32 bits (a float conversion of one word)
    auto unit_cost = [&](uint32_t u, unsigned long long &sum) -> uint32_t {
        unsigned long long v[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t g = 4 * u + k;
            v[k] = gvis[g < groups ? g : groups - 1];  // unconditional: loads stay together
        }
        unsigned long long c = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) c += 4 * u + k < groups ? v[k] : 0ull;
        sum += u < units ? c : 0ull;
        return c > 0xffffffffull ? 0xffffffffu : (uint32_t)c;
    };
    uint32_t cost[kOrderAhead];  // this thread's units t + 1024 i, i < kOrderAhead
    unsigned long long part = 0;
#pragma unroll
    for (uint32_t i = 0; i < kOrderAhead; ++i) cost[i] = unit_cost(t + 1024 * i, part);
    for (uint32_t u = t + 1024 * kOrderAhead; u < units; u += 1024) (void)unit_cost(u, part);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
    if (lane == 0) wsum[wave] = part;
    if (t < kOrderBuckets) base[0][t] = 0;
    lds_barrier();
    unsigned long long total = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) total += wsum[w];
    // bucket = cost in quarters of the mean unit cost (float: any order is
    // a correct one)
    const float scale = total ? 4.0f * (float)units / (float)total : 0.0f;
    auto bucket_of = [&](uint32_t u, uint32_t c) -> uint32_t {
        if (u >= units) return kOrderBuckets;  // no unit
        const float q = (float)c * scale;
        return q >= (float)(kOrderBuckets - 1) ? kOrderBuckets - 1 : (uint32_t)q;
    };
    auto bucket = [&](uint32_t u, uint32_t i) -> uint32_t {
        if (i < kOrderAhead) return bucket_of(u, cost[i]);
        unsigned long long dummy = 0;
        return bucket_of(u, unit_cost(u, dummy));
    };
    // histogram: the lowest lane of each bucket in the wave adds its lanes
    for (uint32_t i = 0; 1024 * i < units; ++i) {
        const uint32_t q = bucket(t + 1024 * i, i);
        const unsigned long long m = bucket_peers(q);
        if (q < kOrderBuckets && (m & below) == 0ull) atomicAdd(&base[0][q], (uint32_t)__popcll(m));
    }
    lds_barrier();
    if (t == 0) {  // bucket starts, heaviest bucket first
        uint32_t run = 0;
        for (int k = (int)kOrderBuckets - 1; k >= 0; --k) {
            const uint32_t c = base[0][k];
            base[0][k] = run;
            run += c;
        }
    }
    lds_barrier();
    // placement, 1024 units a round; wcnt and base alternate by round, so
    // two barriers a round suffice
    for (uint32_t i = 0; 1024 * i < units; ++i) {
        const uint32_t p = i & 1u;
        const uint32_t u = t + 1024 * i;
        const uint32_t q = bucket(u, i);
        if (lane < kOrderBuckets) wcnt[p][wave][lane] = 0;
        const unsigned long long m = bucket_peers(q);
        const uint32_t rank = (uint32_t)__popcll(m & below);
        // the lowest lane of each bucket writes the wave's count (after the
        // zeroing above: one wave's LDS writes complete in order)
        if (q < kOrderBuckets && rank == 0) wcnt[p][wave][q] = (uint32_t)__popcll(m);
        lds_barrier();
        if (q < kOrderBuckets) {
            uint32_t c[16];
#pragma unroll
            for (uint32_t w = 0; w < 16; ++w) c[w] = wcnt[p][w][q];  // all at once
            uint32_t pos = base[p][q] + rank;
#pragma unroll
            for (uint32_t w = 0; w < 16; ++w) pos += w < wave ? c[w] : 0u;
            order[pos] = u;
        }
        if (t < kOrderBuckets) {
            uint32_t c = base[p][t];
#pragma unroll
            for (uint32_t w = 0; w < 16; ++w) c += wcnt[p][w][t];
            base[p ^ 1u][t] = c;
        }
        lds_barrier();
    }
}

// One wave per part of a group: R * 8 of its W targets (walk_group), W / (8 R)
// parts.  Part 0 counts the group's visits and acceptances.
template <int W, int R, bool kWide, bool kDebugAccel>
__global__ __launch_bounds__(256) void bh_walk_kernel(
    const uint32_t *__restrict__ sorted_src, const float2 *__restrict__ pos,
    const float2 *__restrict__ vel, const float4 *__restrict__ node4,
    const uint4 *__restrict__ child, const BhCounters *__restrict__ ctr,
    float2 *__restrict__ pos_out, float2 *__restrict__ vel_out, float2 *__restrict__ acc_dbg,
    uint32_t na, uint32_t cap, float eps2, float theta2, float kv, float kp,
    unsigned long long *__restrict__ gvis, unsigned long long *__restrict__ gacc,
    uint32_t *__restrict__ gchunk, uint32_t xcd, NextKeys nk,
    const uint32_t *__restrict__ order) {
    constexpr uint32_t kParts = W / (8 * R), kLanes = 8 / R;  // lanes that end with a target
    __shared__ WalkShared sh[4];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t b0 = xcd_block(blockIdx.x, gridDim.x, xcd);
    // order: a permutation of the gridDim.x workgroups' units
    const uint32_t b = order ? __builtin_amdgcn_readfirstlane(order[b0]) : b0;
    const uint32_t u = b * 4 + w, g = u / kParts, part = u % kParts;
    if (g >= na / W) return;  // whole wave beyond the last group
    const uint32_t vsrc = sorted_src[g * W + (lane & (W - 1u))];
    const bool real = vsrc < na;  // ForceShader.comp:80-92
    float2 vp = real ? pos[vsrc] : make_float2(0.0f, 0.0f);
    const unsigned long long rb = __ballot(real);
    const uint32_t nreal = (uint32_t)__popcll(W == 64 ? rb : rb & 0xffffffffull);
    // the killed sort last, so the group's first particle is real if any is
    vp.x = real ? vp.x : lane_value(vp.x, 0);
    vp.y = real ? vp.y : lane_value(vp.y, 0);
    // start at the issue priority this group reached in the last step (it
    // gains at W = 64 and nothing at W = 32)
    const uint32_t prio0 = W == 64 ? gchunk[g] / kPrioCarry : 0u;
    const WalkTree tree{node4, child, 0u, uniform(min(ctr->n_nodes, cap)),
                        uniform(ctr->n_in)};
    float ax, ay;
    unsigned long long vis = 0, acc = 0;
    uint32_t chunks = 0;
    walk_group<W, R, kWide>(tree, sh[w], part, vp.x, vp.y, nreal, eps2, theta2, kPrioStepSingle,
                     prio0, ax, ay, vis, acc, chunks);
    if (part == 0 && lane == 0) {  // summed on a dump
        gvis[g] = vis;
        gacc[g] = acc;
        if (W == 64) gchunk[g] = chunks;
    }
    const uint32_t dst = g * W + part * (8 * R) + lane / kLanes;  // slot in the next order
    const uint32_t src = sorted_src[dst];
    if (lane % kLanes != 0u || src >= na) return;
    const float2 p = pos[src], v = vel[src];
    // ForceShader.comp:145-150
    const float nvx = v.x + ax * kv, nvy = v.y + ay * kv;
    const float2 np = make_float2(p.x + (v.x + nvx) * kp, p.y + (v.y + nvy) * kp);
    pos_out[dst] = np;
    vel_out[dst] = make_float2(nvx, nvy);
    if (nk.cells) write_next_key(nk, dst, np);
    if (kDebugAccel) acc_dbg[dst] = make_float2(ax, ay);
}

// 30-bit Morton codes (15 bits per axis) of the same normalised coordinate;
// code >> 10 equals the 20-bit cell because scaling by 32 is exact.
__global__ __launch_bounds__(256) void bh_morton30_kernel(const float2 *__restrict__ pos,
                                                          uint32_t na, uint32_t *__restrict__ out) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= na) return;
    const float2 p = pos[i];
    const float qx = unit_coord(p.x) * 32768.0f, qy = unit_coord(p.y) * 32768.0f;
    uint32_t c = 0xffffffffu;
    if (qx >= 0.0f && qx < 32768.0f && qy >= 0.0f && qy < 32768.0f)
        c = part1by1((uint32_t)qx) | (part1by1((uint32_t)qy) << 1);
    out[i] = c;
}

}  // namespace

size_t bh_capacity(size_t na, uint32_t bits) {
    // every particle plus at most min(4^d, na/2) cells with >= 2 particles per level
    size_t cells = 0;
    for (int d = 0; d <= (int)bits; ++d) {
        const size_t lvl = (size_t)1 << (2 * d);
        cells += lvl < na / 2 ? lvl : na / 2;
    }
    return na + cells + 64;
}

hipError_t bh_alloc(BhBuffers *b, size_t na, uint32_t bits, hipStream_t stream) {
    b->na = na;
    b->bits = bits;
    b->cap = bh_capacity(na, bits);
    b->sort_blocks = sort_tiles(na);
    b->prep_blocks = (na + 255) / 256;
    hipError_t e = hipSuccess;
#define GSIM_ALLOC(ptr, count)                                                  \
    do {                                                                        \
        if (e == hipSuccess) e = hipMalloc((void **)&(ptr), sizeof(*(ptr)) * (count)); \
    } while (0)
    for (int k = 0; k < 2; ++k) {
        GSIM_ALLOC(b->keys[k], na);
        GSIM_ALLOC(b->idx[k], na);
        GSIM_ALLOC(b->cells[k], na);
    }
    // four passes of tile words and group words
    GSIM_ALLOC(b->status, 4 * 256 * (b->sort_blocks + (b->sort_blocks + kLookGroup - 1) / kLookGroup));
    GSIM_ALLOC(b->digit_total, 2 * kDigitCopies * 1024);
    GSIM_ALLOC(b->block_cells, b->prep_blocks);
    GSIM_ALLOC(b->block_leaves, b->prep_blocks);
    GSIM_ALLOC(b->sdep, na + 1);
    GSIM_ALLOC(b->cpos, na);
    GSIM_ALLOC(b->leaf_first, na + 1);
    GSIM_ALLOC(b->leaf_key, na);
    GSIM_ALLOC(b->leaf_sum, na);
    GSIM_ALLOC(b->tile_range, kTileWords);
    GSIM_ALLOC(b->top, kTiles);
    GSIM_ALLOC(b->node4, b->cap);
    GSIM_ALLOC(b->child, b->cap);
    if (bits == kDeepBits) {
        GSIM_ALLOC(b->nsum, b->cap);
        GSIM_ALLOC(b->gran_first, na + 1);
        GSIM_ALLOC(b->gran_key, na);
        GSIM_ALLOC(b->gran_y, na);
        GSIM_ALLOC(b->block_gran, b->prep_blocks);
    }
    GSIM_ALLOC(b->sorted_src, na);
    GSIM_ALLOC(b->ctr, 1);
    GSIM_ALLOC(b->box, 4);
    GSIM_ALLOC(b->box_part, kBoxParts);
    GSIM_ALLOC(b->gchunk, na / 64 + 1);
    GSIM_ALLOC(b->order, na / 128 + 1);
    GSIM_ALLOC(b->gvis, na / 32 + 1);  // one slot per group of W = 32 or 64
    GSIM_ALLOC(b->gacc, na / 32 + 1);
#undef GSIM_ALLOC
    if (e == hipSuccess) e = hipMemsetAsync(b->ctr, 0, sizeof(BhCounters), stream);
    if (e == hipSuccess)
        e = hipMemsetAsync(b->digit_total, 0, sizeof(uint32_t) * 2 * kDigitCopies * 1024, stream);
    if (e == hipSuccess) e = hipMemsetAsync(b->gchunk, 0, sizeof(uint32_t) * (na / 64 + 1), stream);
    if (e == hipSuccess) e = hipMemsetAsync(b->gvis, 0, sizeof(unsigned long long) * (na / 32 + 1), stream);
    if (e == hipSuccess) e = hipMemsetAsync(b->gacc, 0, sizeof(unsigned long long) * (na / 32 + 1), stream);
    if (e == hipSuccess) e = hipMemsetAsync(b->child, 0, sizeof(uint4) * b->cap, stream);
    if (e == hipSuccess) e = hipMemsetAsync(b->node4, 0, sizeof(float4) * b->cap, stream);
    return e;
}

void bh_free(BhBuffers *b) {
    for (int k = 0; k < 2; ++k) {
        (void)hipFree(b->keys[k]);
        (void)hipFree(b->idx[k]);
        (void)hipFree(b->cells[k]);
    }
    void *ptrs[] = {b->status, b->digit_total, b->block_cells, b->block_leaves, b->sdep, b->cpos,
                    b->leaf_first, b->leaf_key, b->leaf_sum, b->tile_range, b->top, b->node4,
                    b->child, b->nsum, b->gran_first, b->gran_key, b->gran_y, b->block_gran,
                    b->sorted_src, b->ctr, b->gchunk, b->order, b->gvis, b->gacc, b->box,
                    b->box_part};
    for (void *p : ptrs) (void)hipFree(p);
    *b = BhBuffers{};
}

// Where this step's walk writes the next build's keys (the buffer the current
// build does not read), or none when the next build must compute them.
static NextKeys next_keys(gsim_sim *s, const uint32_t *perm_out) {
    BhBuffers &b = s->bh;
    if (s->bh_box || !perm_out) return NextKeys{nullptr, nullptr, 0u};
    return NextKeys{perm_out, b.cells[b.kin ^ 1], b.bits == kDeepBits ? 1u : 0u};
}

hipError_t bh_launch_build(gsim_sim *s, const float2 *pos, const float *mass,
                           const uint32_t *perm_in, float2 *pos_out, const float2 *vel,
                           float2 *vel_out, float *mass_out, uint32_t *perm_out) {
    BhBuffers &b = s->bh;
    const uint32_t na = (uint32_t)s->na;
    const bool deep = b.bits == kDeepBits;
    const int bits = (int)b.bits;
    // adaptive box: written by the kernel that makes the keys
    const float *box = s->bh_box ? b.box : nullptr;
    float4 *const box4 = reinterpret_cast<float4 *>(b.box);
    // the sort's input: written by the last walk (fixed domain), else here
    const int kin = b.kin;
    const bool walk = b.walk_keys && !box;
    b.kcells = kin;
    b.sorted_slot = deep ? 1 : 0;
    const uint32_t *sk = b.keys[b.sorted_slot], *si = b.idx[b.sorted_slot];
    const uint32_t pb = (uint32_t)b.prep_blocks;
    const NextKeys nk = next_keys(s, perm_out);
    const EmitArgs emit{pos,       vel,     mass,           perm_in,      pos_out,   vel_out,
                        mass_out,  perm_out, nk.cells,      na,           bits,      b.sdep,
                        b.cpos,    b.leaf_first, b.leaf_key, b.node4,     b.sorted_src, b.ctr,
                        deep ? b.gran_first : nullptr, b.gran_key};
    if (na <= kSmallBuild) {
        uint32_t *const ko = b.keys[b.sorted_slot];
#define GSIM_SMALL(B, D, W)                                                                   \
    bh_small_kernel<B, D, W><<<1, 64 * kSmallWaves, 0, s->stream>>>(emit, b.cells[kin], ko,    \
                                                                    b.tile_range, box4)
        if (box) { if (deep) GSIM_SMALL(true, true, false); else GSIM_SMALL(true, false, false); }
        else if (walk) { if (deep) GSIM_SMALL(false, true, true); else GSIM_SMALL(false, false, true); }
        else { if (deep) GSIM_SMALL(false, true, false); else GSIM_SMALL(false, false, false); }
#undef GSIM_SMALL
    } else {
        // one tile per workgroup, in the keys kernel and in every pass; each
        // pass's status holds its tile words, then its group words
        const uint32_t nblk = (uint32_t)sort_tiles(na);
        const uint32_t nparts = std::min<uint32_t>((na + 255) / 256, kBoxParts);
        if (box) bh_box_partial_kernel<<<nparts, 256, 0, s->stream>>>(pos, na, b.box_part);
        const uint32_t pass_words = (nblk + (nblk + kLookGroup - 1) / kLookGroup) * 256u;
        const int passes = deep ? 4 : 3;
        const uint32_t status_words = (uint32_t)passes * pass_words;
        // digit totals alternate between two halves by build parity
        uint32_t *const totals = b.digit_total + kDigitCopies * 1024 * b.parity;
        uint32_t *const totals_next = b.digit_total + kDigitCopies * 1024 * (b.parity ^ 1u);
        b.parity ^= 1u;
        // 20-bit keys: cells[kin] -> keys[0] -> keys[1] -> keys[0]; 30-bit keys take
        // a fourth pass -> keys[1].  cells[kin] keeps the per-particle cells.
        const int in_of[4] = {-1, 0, 1, 0}, out_of[4] = {0, 1, 0, 1};
#define GSIM_KEYS(R, B, D, W)                                                                  \
    bh_keys_kernel<B, D, R, W><<<nblk, kSortThreads, 0, s->stream>>>(                           \
        pos, perm_in, na, b.cells[kin], b.tile_range, totals, totals_next, b.status,           \
        status_words, b.box_part, nparts, box4)
#define GSIM_SORT(R)                                                                           \
    do {                                                                                       \
        if (box) { if (deep) GSIM_KEYS(R, true, true, false); else GSIM_KEYS(R, true, false, false); } \
        else if (walk) { if (deep) GSIM_KEYS(R, false, true, true); else GSIM_KEYS(R, false, false, true); } \
        else { if (deep) GSIM_KEYS(R, false, true, false); else GSIM_KEYS(R, false, false, false); } \
        for (int pass = 0; pass < passes; ++pass) {                                            \
            const int i = in_of[pass], o = out_of[pass];                                       \
            radix_onesweep_kernel<R><<<nblk, kSortThreads, 0, s->stream>>>(                    \
                i < 0 ? nullptr : b.keys[i], i < 0 ? nullptr : b.idx[i],                       \
                i < 0 ? b.cells[kin] : nullptr, b.keys[o], b.idx[o], na, 8u * pass,            \
                totals + 256 * pass, b.status + (size_t)pass * pass_words, &b.ctr->sort_stall); \
        }                                                                                      \
    } while (0)
        const uint32_t rounds = sort_rounds(na);
        if (rounds == 2) GSIM_SORT(2);
        else if (rounds == 4) GSIM_SORT(4);
        else GSIM_SORT(8);
#undef GSIM_SORT
#undef GSIM_KEYS
        bh_prep_kernel<<<pb, 256, 0, s->stream>>>(sk, na, bits, b.block_cells, b.block_leaves,
                                                  deep ? b.block_gran : nullptr);
        bh_emit_kernel<<<pb, 256, 0, s->stream>>>(sk, si, emit, b.block_cells, b.block_leaves,
                                                  deep ? b.block_gran : nullptr);
    }
    const uint32_t lb = pb < kLeafBlocks ? pb : kLeafBlocks;
    bh_leaf_kernel<<<lb, 256, 0, s->stream>>>(b.leaf_first, b.leaf_key, b.cpos, b.ctr, bits,
                                              b.leaf_sum, b.tile_range, b.node4, b.child,
                                              deep ? b.nsum : nullptr, box);
    if (deep) {
        // sparse levels below depth 10, then depth-10 records for the dense path
        for (int d = (int)kDeepBits - 1; d > (int)kTreeDepth; --d)
            bh_level_kernel<<<pb, 256, 0, s->stream>>>(sk, b.sdep, b.cpos, b.ctr, b.node4,
                                                       b.child, b.nsum, d, box);
        bh_gran_kernel<<<pb, 256, 0, s->stream>>>(sk, b.sdep, b.cpos, b.ctr, b.node4, b.child,
                                                  b.nsum, b.gran_first, b.gran_key, b.leaf_sum,
                                                  b.gran_y, b.tile_range, box);
        bh_tile_kernel<<<kTiles, 256, 0, s->stream>>>(b.tile_range, b.gran_first, b.gran_key,
                                                      b.leaf_sum, b.sdep, b.cpos, b.node4,
                                                      b.child, b.top, box, b.gran_y);
    } else {
        bh_tile_kernel<<<kTiles, 256, 0, s->stream>>>(b.tile_range, b.leaf_first, b.leaf_key,
                                                      b.leaf_sum, b.sdep, b.cpos, b.node4,
                                                      b.child, b.top, box, nullptr);
    }
    return hipGetLastError();
}

uint32_t walk_parts(const gsim_sim *s) {
    const uint32_t groups = (uint32_t)(s->na / s->W), most = s->W / 8;
    if (groups > kWalkSplitGroups) return 1;
    uint32_t parts = 2;
    while (parts < most && 2 * parts * groups <= kWalkFillWaves) parts *= 2;
    return parts;
}

// The walk's workgroup order (null: index order), re-planned from the
// last walk's costs every kOrderReplan steps (costs change slowly) and on
// every trial step, on the walk's own stream: a plan on the side stream
// beside the build measured slower (the cross-stream fork and join cost more
// than the plan).
static const uint32_t *launch_order(gsim_sim *s, uint32_t groups) {
    BhBuffers &b = s->bh;
    if (!s->trav_order) return nullptr;
    if (!b.order_valid || s->order_fresh || s->steps % kOrderReplan == 0) {
        bh_order_plan_kernel<<<1, 1024, 0, s->stream>>>(b.gvis, groups, b.order);
        b.order_valid = s->steps > 0;  // the first step's plan has no costs yet
    }
    return b.order;
}

hipError_t bh_launch_traverse(gsim_sim *s, const float2 *pos, const float2 *vel,
                              float2 *pos_out, float2 *vel_out, const uint32_t *perm_out) {
    BhBuffers &b = s->bh;
    const uint32_t na = (uint32_t)s->na;
    const NextKeys nk = next_keys(s, perm_out);
    // the next build reads the cells this walk writes
    b.walk_keys = nk.cells != nullptr;
    if (b.walk_keys) b.kin ^= 1;
    const bool dbg = (s->debug_flags & GSIM_DEBUG_ACCEL) != 0;
    float2 *acc = dbg ? s->accel : nullptr;
    const uint32_t groups = na / s->W, parts = walk_parts(s);
    const uint32_t grid = (groups * parts + 3) / 4;
    const uint32_t *order = parts == 1 ? launch_order(s, groups) : nullptr;
    const bool wide = b.cap >= s->narrow_nodes;
#define GSIM_WALK(W, R)                                                                        \
    do {                                                                                       \
        auto *k = dbg ? (wide ? bh_walk_kernel<W, R, true, true> : bh_walk_kernel<W, R, false, true>) \
                      : (wide ? bh_walk_kernel<W, R, true, false> : bh_walk_kernel<W, R, false, false>); \
        k<<<grid, 256, 0, s->stream>>>(b.sorted_src, pos, vel, b.node4, b.child, b.ctr,        \
                                       pos_out, vel_out, acc, na, (uint32_t)b.cap, s->eps2,    \
                                       s->theta2, s->kv, s->kp, b.gvis, b.gacc, b.gchunk,      \
                                       s->xcd_order, nk, order);                               \
    } while (0)
    if (s->W == 64) {
        if (parts == 1) GSIM_WALK(64, 8);
        else if (parts == 2) GSIM_WALK(64, 4);
        else if (parts == 4) GSIM_WALK(64, 2);
        else GSIM_WALK(64, 1);
    } else {
        if (parts == 1) GSIM_WALK(32, 4);
        else if (parts == 2) GSIM_WALK(32, 2);
        else GSIM_WALK(32, 1);
    }
#undef GSIM_WALK
    return hipGetLastError();
}

hipError_t bh_launch_morton30(gsim_sim *s, const float2 *pos, uint32_t *out) {
    const uint32_t na = (uint32_t)s->na;
    bh_morton30_kernel<<<(na + 255) / 256, 256, 0, s->stream>>>(pos, na, out);
    return hipGetLastError();
}

}  // namespace gsim
