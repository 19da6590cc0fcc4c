// Device helpers shared by the single-system and batched Barnes-Hut kernels.
#pragma once

#include "internal.hpp"
#include "lane_ops.hpp"

namespace gsim {

__device__ __forceinline__ uint32_t part1by1(uint32_t v) {
    v = (v | (v << 8)) & 0x00ff00ffu;
    v = (v | (v << 4)) & 0x0f0f0f0fu;
    v = (v | (v << 2)) & 0x33333333u;
    v = (v | (v << 1)) & 0x55555555u;
    return v;
}

// (p / S + 1) * 0.5, the normalised coordinate of InitShader.comp:80.
// Division is IEEE (no reciprocal contraction); the file is built with
// -ffp-contract=off, so each operation rounds as written.
__device__ __forceinline__ float unit_coord(float p) { return ((p / kSimSize) + 1.0f) * 0.5f; }

// A workgroup barrier that orders LDS only: __syncthreads() also waits for
// the wave's outstanding global stores, which costs a store's latency at
// every barrier that follows one.  For barriers that guard LDS data alone.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ uint32_t cell20(float x, float y) {
    const float qx = unit_coord(x) * (float)kTreeSize;
    const float qy = unit_coord(y) * (float)kTreeSize;
    if (qx >= 0.0f && qx < (float)kTreeSize && qy >= 0.0f && qy < (float)kTreeSize)
        return part1by1((uint32_t)qx) | (part1by1((uint32_t)qy) << 1);
    return 0xffffffffu;
}

// Depth of the deepest cell shared by two in-domain cells (0..10).
__device__ __forceinline__ int shared_depth(uint32_t a, uint32_t b) {
    const uint32_t x = a ^ b;
    if (x == 0) return 10;
    return 9 - ((31 - __clz(x)) >> 1);
}

// The same for keys of `bits` bits per axis (0..bits).
__device__ __forceinline__ int shared_depth_bits(uint32_t a, uint32_t b, int bits) {
    const uint32_t x = a ^ b;
    if (x == 0) return bits;
    return bits - 1 - ((31 - __clz(x)) >> 1);
}

// 15-bit cells (30-bit keys): the normalised coordinate of cell20 scaled by
// 32768 instead of 1024.  Scaling by a power of two is exact, so key >> 10 is
// the 20-bit cell.
__device__ __forceinline__ uint32_t cell30(float x, float y) {
    const float qx = unit_coord(x) * 32768.0f, qy = unit_coord(y) * 32768.0f;
    if (qx >= 0.0f && qx < 32768.0f && qy >= 0.0f && qy < 32768.0f)
        return part1by1((uint32_t)qx) | (part1by1((uint32_t)qy) << 1);
    return 0xffffffffu;
}

// Workgroups of a launch are dispatched to the 8 XCDs round-robin (workgroup
// b to XCD b mod 8), and each XCD has its own L2.  xcd_block renumbers them so
// that XCD x runs runs of c consecutive logical workgroups (logical blocks
// [8ck + cx, 8ck + cx + c) for k = 0, 1, ...), spatially adjacent groups,
// which walk nearly the same cells and leaf runs, then sharing an L2; the
// last nb mod 8c workgroups keep their number.  From 8c >= nb on, each XCD
// takes one contiguous range (q or q + 1 workgroups for nb = 8q + r).
// c <= 1 is the plain round-robin order.  A bijection on [0, nb).
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb, uint32_t c) {
    if (c <= 1u) return b;
    const uint32_t x = b & 7u, i = b >> 3;
    if (8u * c >= nb) {
        const uint32_t q = nb >> 3, r = nb & 7u;
        return x * q + min(x, r) + i;
    }
    const uint32_t span = 8u * c, whole = nb / span * span;
    if (b >= whole) return b;
    return (i / c) * span + x * c + i % c;
}

// Radius base of the fixed domain: S*S*2 (TreeMoveShader.comp:70-71).
constexpr float kFixedR0 = kSimSize * kSimSize * 2.0f;

// r0 / 4^d: S*S*2 / 4^d for the fixed domain, (h*h)*2 / 4^d for the adaptive
// box; exact in FP32 (division by a power of two).
__device__ __forceinline__ float cell_radius(int d, float r0) {
    return r0 / (float)(1u << (2 * d));
}

// Adaptive box {cx, cy, h, r0}: ((p - c) / h + 1) * 0.5 * 1024, clamped to
// [0, 1023]; only non-finite positions are outside.
__device__ __forceinline__ uint32_t cell20_box(float x, float y, float cx, float cy, float h) {
    if (!__builtin_isfinite(x) || !__builtin_isfinite(y)) return 0xffffffffu;
    const float qx = ((((x - cx) / h) + 1.0f) * 0.5f) * (float)kTreeSize;
    const float qy = ((((y - cy) / h) + 1.0f) * 0.5f) * (float)kTreeSize;
    const uint32_t ix = min(qx > 0.0f ? (uint32_t)qx : 0u, kTreeSize - 1);
    const uint32_t iy = min(qy > 0.0f ? (uint32_t)qy : 0u, kTreeSize - 1);
    return part1by1(ix) | (part1by1(iy) << 1);
}

// cell20_box on the 32768^2 grid (clamped to [0, 32767]).
__device__ __forceinline__ uint32_t cell30_box(float x, float y, float cx, float cy, float h) {
    if (!__builtin_isfinite(x) || !__builtin_isfinite(y)) return 0xffffffffu;
    const float qx = ((((x - cx) / h) + 1.0f) * 0.5f) * 32768.0f;
    const float qy = ((((y - cy) / h) + 1.0f) * 0.5f) * 32768.0f;
    const uint32_t ix = min(qx > 0.0f ? (uint32_t)qx : 0u, 32767u);
    const uint32_t iy = min(qy > 0.0f ? (uint32_t)qy : 0u, 32767u);
    return part1by1(ix) | (part1by1(iy) << 1);
}

__device__ __forceinline__ void accumulate(float nx, float ny, float m, float px, float py,
                                           float eps2, float &ax, float &ay) {
    const float dx = nx - px, dy = ny - py;
    const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, eps2));
    const float inv = __builtin_amdgcn_rsqf(r2);
    const float s = (m * inv) * (inv * inv);
    ax = __builtin_fmaf(dx, s, ax);
    ay = __builtin_fmaf(dy, s, ay);
}

__device__ __forceinline__ TileCell reduce4(const TileCell &a, const TileCell &b,
                                            const TileCell &c, const TileCell &d) {
    TileCell r;
    r.n = a.n + b.n + c.n + d.n;
    r.y = a.y + b.y + c.y + d.y;
    r.y += r.y > 1u ? 1u : 0u;  // TreeInitShader.comp:83
    r.f = min(min(a.f, b.f), min(c.f, d.f));
    r.pad = 0;
    r.sx = ((a.sx + b.sx) + c.sx) + d.sx;  // TreeInitShader.comp:79-80
    r.sy = ((a.sy + b.sy) + c.sy) + d.sy;
    r.sm = ((a.sm + b.sm) + c.sm) + d.sm;
    r.pad2 = 0.0f;
    return r;
}

// The depth-d cell node c (first particle c.f) at its pre-order slot, given,
// with its children's subtree sizes (kLeafMark: a leaf cell's particles).
__device__ __forceinline__ void emit_cell_at(const TileCell &c, int d, uint32_t slot, uint4 sizes,
                                             float4 *__restrict__ node4,
                                             uint4 *__restrict__ child, float r0 = kFixedR0) {
    if (c.y <= 1u) return;
    float px = c.sx, py = c.sy;
    if (c.sm != 0.0f) {  // TreeMoveShader.comp:66-67
        px = px / c.sm;
        py = py / c.sm;
    }
    child[slot] = sizes;
    node4[slot] = make_float4(px, py, c.sm, cell_radius(d, r0));
}

// Depth d of the cell starting at sorted position f: slot f + C(f) + (d - s(f) - 1).
__device__ __forceinline__ uint32_t cell_slot(uint32_t f, int d, const int8_t *__restrict__ sdep,
                                              const uint32_t *__restrict__ cpos) {
    return f + cpos[f] + (uint32_t)(d - (int)sdep[f] - 1);
}

__device__ __forceinline__ void emit_cell(const TileCell &c, int d, uint4 sizes,
                                          const int8_t *__restrict__ sdep,
                                          const uint32_t *__restrict__ cpos,
                                          float4 *__restrict__ node4, uint4 *__restrict__ child,
                                          float r0 = kFixedR0) {
    if (c.y <= 1u) return;
    emit_cell_at(c, d, cell_slot(c.f, d, sdep, cpos), sizes, node4, child, r0);
}

// The subtree sizes of four sibling cells.
__device__ __forceinline__ uint4 sizes4(const TileCell *c) {
    return make_uint4(c[0].y, c[1].y, c[2].y, c[3].y);
}

// Words shared by workgroups of one launch, on any XCD.
__device__ __forceinline__ uint32_t status_load(const uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void status_store(uint32_t *p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- dense reduction of a depth-5 tile, and of the top --------------------------

// Level offsets inside `up`: depth 9 at 0 (256 cells), 8 at 256 (64),
// 7 at 320 (16), 6 at 336 (4), 5 at 340 (1).
__device__ __forceinline__ int tile_level_offset(int d) {
    return d == 9 ? 0 : d == 8 ? 256 : d == 7 ? 320 : d == 6 ? 336 : 340;
}

// A tile's record for the workgroup that reduces the top, on any XCD: each
// word is stored at the scope of the device and has arrived before the call
// returns, and is loaded at that scope, past the XCD's own L2.  A fence would
// write that whole L2 back, once a tile.
// The order comes from the machine, not from the language, whose relaxed
// accesses promise it for one word only.  It rests on the memory model of
// gfx940 to gfx950 (LLVM's AMDGPU guide): a store with sc1, which a store at
// device scope is, writes through the L2, and vmcnt counts it off once it is
// visible to the device, so s_waitcnt vmcnt(0) before the counter's atomic
// orders the two, as a release at that scope does for its own write-back; the
// reader's loads with sc1 are issued after the counter's value has returned
// (it decides the branch that leads to them) and take no line of their L2.
__device__ __forceinline__ void publish_top(TileCell *to, const TileCell &c) {
    uint32_t *w = reinterpret_cast<uint32_t *>(to);
    status_store(w + 0, c.n);
    status_store(w + 1, c.y);
    status_store(w + 2, c.f);
    status_store(w + 4, __float_as_uint(c.sx));
    status_store(w + 5, __float_as_uint(c.sy));
    status_store(w + 6, __float_as_uint(c.sm));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

__device__ __forceinline__ TileCell published_top(const TileCell *from) {
    const uint32_t *w = reinterpret_cast<const uint32_t *>(from);
    TileCell c;
    c.n = status_load(w + 0);
    c.y = status_load(w + 1);
    c.f = status_load(w + 2);
    c.pad = 0u;
    c.sx = __uint_as_float(status_load(w + 4));
    c.sy = __uint_as_float(status_load(w + 5));
    c.sm = __uint_as_float(status_load(w + 6));
    c.pad2 = 0.0f;
    return c;
}

// One occupied depth-5 tile T of a tree, by one workgroup (leaves [lb, le) of
// its range; tile_range: the tree's kTileWords).  leaf_y (15-bit leaves): the
// depth-10 records are granules whose subtree size is given; otherwise leaves
// of n particles, y = n + [n >= 2].  The depth-10 nodes themselves are already
// written.
// The last occupied tile's workgroup to finish also reduces the 1024 depth-5
// cells to the root and writes depths 4..0, so the top needs no launch of its
// own.  Occupied tiles publish their record, then count themselves done in
// their group of 32 tiles; the last of a group counts the group done, and the
// last group's workgroup goes on.  How many to expect is read from tile_range.
// One counter for all tiles is a chain of 1024 same-address atomics across the
// XCDs, and the fence it needs writes an L2 back for each.  Empty tiles have
// no workgroup here; their empty record comes from tile_range.
// Bound by latency: its chain of loads, six levels and two counts.  53.3 ->
// 14.5 us with every tile occupied (200,000 particles, adaptive box), 12.7 ->
// 8.1 us at 500,000 in the fixed domain, 16.3 -> 8.2 us at 5,000: the counters
// a cache line apart 57 -> 22, the smaller LDS image and the loads ahead of it
// the rest.
struct TileShared {
    // the depth-10 cells {sums, particles} and {subtree size, first particle}:
    // 35 KB with `up`, so all 1024 workgroups of a tree are resident (four a CU)
    float4 sum10[1024];
    uint2 yf10[1024];
    TileCell up[341];
    uint32_t last, wave_groups[4];
};

__device__ __forceinline__ void reduce_tile(
    uint32_t T, uint32_t *__restrict__ tile_range, const uint32_t *__restrict__ leaf_first,
    const uint32_t *__restrict__ leaf_key, const float4 *__restrict__ leaf_sum,
    const uint32_t *__restrict__ leaf_y, const int8_t *__restrict__ sdep,
    const uint32_t *__restrict__ cpos, float4 *__restrict__ node4, uint4 *__restrict__ child,
    TileCell *__restrict__ top, float r0, TileShared &sh) {
    const uint32_t t = threadIdx.x;
    const uint32_t lb = tile_range[2 * T], le = tile_range[2 * T + 1];
    uint32_t *const done = tile_range + 2 * kTiles;  // 32 words apart; the groups' last
    const uint2 *const range = reinterpret_cast<const uint2 *>(tile_range);
    uint32_t expect = 0;  // occupied tiles of this tile's group
    if (t >= 192) {  // the wave that publishes: it emits fewest cells
        const uint2 r = range[(T & ~31u) + (t & 31u)];
        expect = (uint32_t)__popcll(__ballot(t < 224 && r.x != r.y));
    }
    // a tile holds at most 1024 leaves (granules): four per thread, loaded
    // together
    struct Leaf {
        float4 s;
        uint32_t k, f, y;
    };
    auto leaf = [&](uint32_t u) {
        const uint32_t L = min(lb + t + 256 * u, le - 1);
        return Leaf{leaf_sum[L], leaf_key[L], leaf_first[L], leaf_y ? leaf_y[L] : 0u};
    };
    const Leaf a0 = leaf(0), a1 = leaf(1), a2 = leaf(2), a3 = leaf(3);
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
        sh.sum10[t + 256 * u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        sh.yf10[t + 256 * u] = make_uint2(0u, 0xffffffffu);
    }
    lds_barrier();
    auto place = [&](uint32_t u, const Leaf &a) {
        if (lb + t + 256 * u >= le) return;
        const uint32_t c = a.k & 1023u, n = __float_as_uint(a.s.w);
        sh.sum10[c] = a.s;
        sh.yf10[c] = make_uint2(leaf_y ? a.y : n + (n >= 2u ? 1u : 0u), a.f);
    };
    place(0, a0);
    place(1, a1);
    place(2, a2);
    place(3, a3);
    lds_barrier();
    auto kid = [&](uint32_t u) {  // of depth-9 cell t
        const float4 s = sh.sum10[4 * t + u];
        const uint2 q = sh.yf10[4 * t + u];
        return TileCell{__float_as_uint(s.w), q.x, q.y, 0u, s.x, s.y, s.z, 0.0f};
    };
    const TileCell k0 = kid(0), k1 = kid(1), k2 = kid(2), k3 = kid(3);
    const uint4 sizes9 = make_uint4(k0.y, k1.y, k2.y, k3.y);
    const TileCell c9 = reduce4(k0, k1, k2, k3);
    sh.up[t] = c9;
    lds_barrier();
    for (int d = 8; d >= 5; --d) {
        const uint32_t cnt = 1u << (2 * (d - 5));
        const int o = tile_level_offset(d), oc = tile_level_offset(d + 1);
        if (t < cnt)
            sh.up[o + t] = reduce4(sh.up[oc + 4 * t], sh.up[oc + 4 * t + 1], sh.up[oc + 4 * t + 2],
                                sh.up[oc + 4 * t + 3]);
        lds_barrier();
    }
    if (t == 192) {
        publish_top(top + T, sh.up[340]);
        sh.last = atomicAdd(done + T / 32 * 32, 1u) + 1u == expect ? 1u : 0u;
    }
    if (t < 85) {  // depths 8..5
        const uint32_t c = 256 + t;
        const int d = c < 320 ? 8 : c < 336 ? 7 : c < 340 ? 6 : 5;
        const TileCell *kids = sh.up + tile_level_offset(d + 1) + 4 * (c - tile_level_offset(d));
        emit_cell(sh.up[c], d, sizes4(kids), sdep, cpos, node4, child, r0);
    }
    emit_cell(c9, 9, sizes9, sdep, cpos, node4, child, r0);
    lds_barrier();
    if (!sh.last) return;
    const uint4 ra = reinterpret_cast<const uint4 *>(tile_range)[2 * t];
    const uint4 rb = reinterpret_cast<const uint4 *>(tile_range)[2 * t + 1];
    const bool in0 = ra.x != ra.y, in1 = ra.z != ra.w, in2 = rb.x != rb.y, in3 = rb.z != rb.w;
    // groups with an occupied tile: eight threads a group, eight groups a wave
    unsigned long long m = __ballot(in0 || in1 || in2 || in3);
    m |= m >> 4;
    m |= m >> 2;
    m |= m >> 1;
    if ((t & 63) == 0)
        sh.wave_groups[t >> 6] = (uint32_t)__popcll(m & 0x0101010101010101ull);
    lds_barrier();
    if (t == 0)
        sh.last = atomicAdd(done + 32 * 32, 1u) + 1u ==
                       sh.wave_groups[0] + sh.wave_groups[1] + sh.wave_groups[2] + sh.wave_groups[3]
                   ? 1u
                   : 0u;
    lds_barrier();
    if (!sh.last) return;
    asm volatile("" ::: "memory");  // holds the compiler to it: counts, then records
    // depths 4..0 in `up` at the offsets of depths 9..5
    const TileCell empty{0u, 0u, 0xffffffffu, 0u, 0.0f, 0.0f, 0.0f, 0.0f};
    const TileCell t0 = in0 ? published_top(top + 4 * t) : empty;
    const TileCell t1 = in1 ? published_top(top + 4 * t + 1) : empty;
    const TileCell t2 = in2 ? published_top(top + 4 * t + 2) : empty;
    const TileCell t3 = in3 ? published_top(top + 4 * t + 3) : empty;
    const TileCell c4 = reduce4(t0, t1, t2, t3);
    sh.up[t] = c4;
    emit_cell(c4, 4, make_uint4(t0.y, t1.y, t2.y, t3.y), sdep, cpos, node4, child, r0);
    lds_barrier();
    for (int d = 3; d >= 0; --d) {
        const uint32_t cnt = 1u << (2 * d);
        const int o = tile_level_offset(d + 5), oc = tile_level_offset(d + 6);
        if (t < cnt)
            sh.up[o + t] = reduce4(sh.up[oc + 4 * t], sh.up[oc + 4 * t + 1], sh.up[oc + 4 * t + 2],
                                sh.up[oc + 4 * t + 3]);
        lds_barrier();
    }
    if (t < 85) {  // depths 3..0
        const uint32_t c = 256 + t;
        const int d = c < 320 ? 3 : c < 336 ? 2 : c < 340 ? 1 : 0;
        const TileCell *kids =
            sh.up + tile_level_offset(d + 6) + 4 * (c - tile_level_offset(d + 5));
        emit_cell(sh.up[c], d, sizes4(kids), sdep, cpos, node4, child, r0);
    }
}

// Exclusive scan of data[0, count) in place by one workgroup of 1024 threads:
// chunks of 4096 values, four consecutive values per thread (coalesced), wave
// shuffles, the 16 wave sums scanned by wave 0, a carry between chunks.
// wsum: 16 words of LDS.
__device__ __forceinline__ void scan_inplace_1024(uint32_t *__restrict__ data, uint32_t count,
                                                  uint32_t *wsum) {
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < count; base += 4096) {
        const uint32_t i0 = base + 4 * t;
        uint32_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = i0 + u < count ? data[i0 + u] : 0u;
        const uint32_t s = (v[0] + v[1]) + (v[2] + v[3]);
        uint32_t x = s;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = __shfl_up(x, off, 64);
            if (lane >= (uint32_t)off) x += y;
        }
        if (lane == 63) wsum[wave] = x;
        lds_barrier();
        if (wave == 0) {
            uint32_t w = lane < 16 ? wsum[lane] : 0u;
#pragma unroll
            for (int off = 1; off < 16; off <<= 1) {
                const uint32_t y = __shfl_up(w, off, 64);
                if (lane >= (uint32_t)off) w += y;
            }
            if (lane < 16) wsum[lane] = w;
        }
        lds_barrier();
        uint32_t run = carry + (wave ? wsum[wave - 1] : 0u) + (x - s);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (i0 + u < count) data[i0 + u] = run;
            run += v[u];
        }
        carry += wsum[15];
        lds_barrier();  // wsum is rewritten by the next chunk
    }
}

// Inclusive scan of one value across a 256-thread workgroup; returns the
// inclusive prefix and writes the workgroup total.
__device__ __forceinline__ uint32_t block_scan256(uint32_t x, uint32_t *total,
                                                  uint32_t *wsum /* [4] LDS */) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = __shfl_up(x, off, 64);
        if (lane >= (uint32_t)off) x += u;
    }
    if (lane == 63) wsum[wave] = x;
    lds_barrier();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; ++w) before += wsum[w];
    *total = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    lds_barrier();
    return x + before;
}

// Inclusive wave scan of two counters.
__device__ __forceinline__ void wave_scan2(uint32_t &a, uint32_t &b) {
    const uint32_t lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t ua = __shfl_up(a, off, 64);
        const uint32_t ub = __shfl_up(b, off, 64);
        if (lane >= (uint32_t)off) {
            a += ua;
            b += ub;
        }
    }
}

// ---- leaf sums: m*x, m*y, m of a leaf's particles in ascending sorted order --
// A leaf's particle nodes are consecutive, [f, e) of node4: their products
// (pos *= mass, InitShader.comp:102) are formed here.  Both forms add the
// products one after another in the same order, so a leaf gets the same bits
// whichever sums it.

// Leaves of at most kSmallLeaf particles are summed by one lane.
constexpr uint32_t kSmallLeaf = 24;

// Loads go out eight at a time (one round trip per eight products); the
// additions keep the sequential order.
__device__ __forceinline__ float4 lane_leaf_sum(const float4 *__restrict__ node4, uint32_t f,
                                                uint32_t e) {
    typedef float v4 __attribute__((ext_vector_type(4)));  // stays in registers
    const v4 *vp = reinterpret_cast<const v4 *>(node4);
    const v4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float sx = 0.0f, sy = 0.0f, sm = 0.0f;
    for (uint32_t k = f; k < e; k += 8) {
        v4 q[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) q[u] = k + u < e ? vp[k + u] : zero;
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            const bool in = k + u < e;
            sx = in ? sx + q[u].x * q[u].z : sx;
            sy = in ? sy + q[u].y * q[u].z : sy;
            sm = in ? sm + q[u].z : sm;
        }
    }
    return make_float4(sx, sy, sm, 0.0f);
}

// A larger leaf [f, e) (wave-uniform bounds) by the whole wave: 64 products
// per coalesced load, four chunks in flight ahead of the one being summed,
// staged in the wave's LDS component by component (64 m*x, 64 m*y, 64 m).
// Lanes 0, 1 and 2 each sum one component, reading it 16 bytes at a time, so
// the wave issues one add per product; each component's order is the leaf's
// particle order, from +0.  The dependent chain of adds is what remains.
__device__ __forceinline__ float4 wave_leaf_sum(float4 *stage, const float4 *__restrict__ node4,
                                                uint32_t f, uint32_t e, uint32_t lane) {
    typedef float v4 __attribute__((ext_vector_type(4)));  // stays in registers
    const v4 *vp = reinterpret_cast<const v4 *>(node4);
    float *st = reinterpret_cast<float *>(stage);
    const uint32_t comp = lane < 3u ? lane : 0u;  // the component this lane sums
    const v4 *sc = reinterpret_cast<const v4 *>(st + 64 * comp);
    float s = 0.0f;
    // loads past the leaf read its last record instead (never summed): no
    // lane-dependent branch, so each wait is for the one chunk it needs
    v4 q[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) q[u] = vp[min(f + 64 * u + lane, e - 1)];
    for (uint32_t base = f; base < e; base += 256) {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t cb = base + 64 * u;
            if (cb >= e) break;
            st[lane] = q[u].x * q[u].z;
            st[64 + lane] = q[u].y * q[u].z;
            st[128 + lane] = q[u].z;
            __builtin_amdgcn_wave_barrier();
            q[u] = vp[min(cb + 256 + lane, e - 1)];
            const uint32_t cnt = min(64u, e - cb);
            if (cnt == 64u) {
#pragma unroll
                for (int h = 0; h < 16; h += 4) {
                    v4 r[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) r[j] = sc[h + j];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        s = s + r[j].x;
                        s = s + r[j].y;
                        s = s + r[j].z;
                        s = s + r[j].w;
                    }
                }
            } else {
                for (uint32_t k = 0; k < cnt; ++k) s = s + st[64 * comp + k];
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    return make_float4(__shfl(s, 0, 64), __shfl(s, 1, 64), __shfl(s, 2, 64), 0.0f);
}

// ---- the walk of one vote group --------------------------------------------
// A vote group is W = 64 or 32 consecutive sorted particles that take every
// cell together (ForceShader.comp:111-141): a cell is accepted iff every real
// particle has radius <= (dx*dx + dy*dy + eps2) * theta2, rounded as the
// shader writes it, and opened otherwise; particles are always accepted.
//
// One wave walks the cells 64 at a time, one per lane, from a stack in LDS.
// Rounding is monotonic, so the shader's own expression at the nearest point
// of the group's bounding box is a lower bound of every particle's value: a
// cell whose radius is within it is accepted by all, and the others are voted
// on, eight at a time.  The accepted set is therefore the shader's, exactly.
// An opened cell pushes its children (their slots follow from their subtree
// sizes, `child`); an opened leaf cell and every accepted node append their
// slots to the list of sources.
//
// The sources are summed eight at a time: lane = 8 * slot + stream holds
// R targets (t = slot * R + r) and sums every eighth source (its stream) for
// each, straight from the node records; at the end a target's eight streams
// are added in a fixed order.  A target's sum depends only on the order of
// the list, so the same group gives the same bits whichever R its targets
// are dealt to waves by.
//
// What bounds it: the VALU, 9 operations (a SIMD issues one every 2 clocks from
// two waves in turn where all operands are vector registers, otherwise one
// every 4) and one v_rsq_f32 (8 to 12 clocks) per source and target.  They are
// kept in the order written: interleaved over pairs by the compiler the same
// operations took 43 clocks a pair, in sequence 34-37 (500,000 particles, W =
// 32: 226 against 199 us).  Matrix instructions for the differences bring
// nothing: v_mfma_f32_32x32x2_f32 holds up the VALU for as long as the
// subtractions it saves.  Measured against one cell at a time per wave, with
// runs staged in LDS (us per walk): 500,000 particles at W = 32 214 -> 176, a
// million at W = 64 929 -> 881, 200,017 with 15-bit leaves 124 -> 39, 5,003 at
// theta 0.5 109 -> 25.

// Cells pushed but not yet visited, and sources not yet summed, of one wave.
// Visiting n cells pushes at most 4 n, so n is kept small enough to leave
// kWalkMargin free, more than the 3 entries a level that visiting one cell at
// a time can add down to depth 15.
constexpr uint32_t kWalkStack = 512;
constexpr uint32_t kWalkList = 512;
constexpr uint32_t kWalkMargin = 64;
struct WalkShared {
    uint4 list4[kWalkList / 4];
    uint32_t stack[kWalkStack + 64];  // a read of 64 entries may start at any of them
    float4 cell[64];                  // cells being voted on
};

// Orders one wave's LDS accesses (a wave's LDS operations complete in order:
// this holds the compiler to it).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint32_t uniform(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}

__device__ __forceinline__ uint32_t lane_rank(unsigned long long m) {  // set bits below this lane
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ float lane_value(float v, uint32_t lane) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}

// Minimum (kMax: maximum) over the wave, in every lane.
template <bool kMax>
__device__ __forceinline__ float wave_extreme(float v) {
    auto op = [](float a, float b) { return kMax ? fmaxf(a, b) : fminf(a, b); };
    v = op(v, dpp<kDppXor1>(v));
    v = op(v, dpp<kDppXor2>(v));
    v = op(v, dpp<kDppXor7>(v));
    v = op(v, dpp<kDppXor15>(v));
    v = op(v, __shfl_xor(v, 16, 64));
    return op(v, __shfl_xor(v, 32, 64));
}

// The (x, y, mass) words of a node record.
typedef float f3v __attribute__((ext_vector_type(3)));

struct BoxXY {
    float x0, x1, y0, y1;
};

// One source (x, y, mass) against this lane's targets.
template <int R>
__device__ __forceinline__ void add_source(f3v q, const float (&tx)[R], const float (&ty)[R],
                                           float eps2, float (&ax)[R], float (&ay)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        accumulate(q.x, q.y, q.z, tx[r], ty[r], eps2, ax[r], ay[r]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// A list entry: the byte offset of the node's record, or with kWide (trees
// that reach beyond 4 GiB of records, kNarrowNodes) its slot.
template <bool kWide>
__device__ __forceinline__ uint32_t source_key(uint32_t slot) {
    return kWide ? slot : slot * 16u;
}

template <bool kWide>
__device__ __forceinline__ f3v load_source(const float4 *__restrict__ node4, uint32_t key) {
    const float *p = kWide ? reinterpret_cast<const float *>(node4 + key)
                           : reinterpret_cast<const float *>(
                                 reinterpret_cast<const char *>(node4) + key);
    f3v r;
    r.x = p[0];
    r.y = p[1];
    r.z = p[2];
    return r;
}

// Record `slot` of an array of 16-byte records.
template <bool kWide, typename T>
__device__ __forceinline__ T tree_record(const T *__restrict__ base, uint32_t slot) {
    static_assert(sizeof(T) == 16, "16-byte records");
    return kWide ? base[slot]
                 : *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + slot * 16u);
}

// The whole blocks of 32 of the first list entries: stream s takes entries
// 4s .. 4s + 3 of each.  Two sources a stream are loaded while the two before
// are summed, their list entries one block earlier.  A walk of 500,000
// particles (galaxy, W = 64): 232 us; four sources at a time (24 registers
// instead of 12) 245, the entries read when needed 236, one source at a time
// 243.
template <int R, bool kWide>
__device__ __forceinline__ void sum_blocks(const WalkShared &sh, uint32_t blocks, uint32_t stream,
                                           const float4 *__restrict__ node4, const float (&tx)[R],
                                           const float (&ty)[R], float eps2, float (&ax)[R],
                                           float (&ay)[R]) {
    if (!blocks) return;
    const uint2 *const pairs = reinterpret_cast<const uint2 *>(sh.list4) + 2 * stream;
    uint2 k = pairs[0], kn = pairs[1];
    f3v a0 = load_source<kWide>(node4, k.x), a1 = load_source<kWide>(node4, k.y);
    for (uint32_t b = 0; b < blocks; ++b) {
        const f3v c0 = load_source<kWide>(node4, kn.x), c1 = load_source<kWide>(node4, kn.y);
        k = pairs[16 * min(b + 1, blocks - 1)];
        add_source<R>(a0, tx, ty, eps2, ax, ay);
        add_source<R>(a1, tx, ty, eps2, ax, ay);
        a0 = load_source<kWide>(node4, k.x);
        a1 = load_source<kWide>(node4, k.y);
        kn = pairs[16 * min(b + 1, blocks - 1) + 1];
        add_source<R>(c0, tx, ty, eps2, ax, ay);
        add_source<R>(c1, tx, ty, eps2, ax, ay);
    }
}

// The last count < 32 entries, stream s taking entry 8 j + s of each eight; a
// stream without one adds a massless source far away (exactly nothing).
template <int R, bool kWide>
__device__ __forceinline__ void sum_rest(const WalkShared &sh, uint32_t first, uint32_t count,
                                         uint32_t stream, const float4 *__restrict__ node4,
                                         const float (&tx)[R], const float (&ty)[R], float eps2,
                                         float (&ax)[R], float (&ay)[R]) {
    const uint32_t *list = reinterpret_cast<const uint32_t *>(sh.list4);
    for (uint32_t j = 0; j < count; j += 8) {
        const bool in = j + stream < count;
        f3v q = load_source<kWide>(node4, list[first + (in ? j + stream : j)]);
        q.x = in ? q.x : 1e18f;
        q.z = in ? q.z : 0.0f;
        add_source<R>(q, tx, ty, eps2, ax, ay);
    }
}

// The sum of a target's eight streams: the lanes of a slot exchange with
// stream ^ 7, ^ 2 and ^ 1, halving the targets each still holds, so that lane
// l ends with target l / (8 / R) and the order of additions is the same for
// every R.
template <int R>
__device__ __forceinline__ float sum_streams(const float (&a)[R], uint32_t lane) {
    if constexpr (R == 8) {
        float b[4];
        const bool up = (lane & 4u) != 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            b[i] = (up ? a[i + 4] : a[i]) + dpp<kDppXor7>(up ? a[i] : a[i + 4]);
        const bool u2 = (lane & 2u) != 0;
        const float c0 = (u2 ? b[2] : b[0]) + dpp<kDppXor2>(u2 ? b[0] : b[2]);
        const float c1 = (u2 ? b[3] : b[1]) + dpp<kDppXor2>(u2 ? b[1] : b[3]);
        const bool u1 = (lane & 1u) != 0;
        return (u1 ? c1 : c0) + dpp<kDppXor1>(u1 ? c0 : c1);
    } else if constexpr (R == 4) {
        const bool up = (lane & 4u) != 0, u2 = (lane & 2u) != 0;
        const float b0 = (up ? a[2] : a[0]) + dpp<kDppXor7>(up ? a[0] : a[2]);
        const float b1 = (up ? a[3] : a[1]) + dpp<kDppXor7>(up ? a[1] : a[3]);
        const float c = (u2 ? b1 : b0) + dpp<kDppXor2>(u2 ? b0 : b1);
        return c + dpp<kDppXor1>(c);
    } else if constexpr (R == 2) {
        const bool up = (lane & 4u) != 0;
        const float b = (up ? a[1] : a[0]) + dpp<kDppXor7>(up ? a[0] : a[1]);
        const float c = b + dpp<kDppXor2>(b);
        return c + dpp<kDppXor1>(c);
    } else {
        static_assert(R == 1, "targets per lane");
        const float b = a[0] + dpp<kDppXor7>(a[0]);
        const float c = b + dpp<kDppXor2>(b);
        return c + dpp<kDppXor1>(c);
    }
}

// Issue priority of a walking wave: dense-core groups are the tail of a
// launch whose groups are all resident from the start, so a wave rises one
// level (s_setprio 1..3) per prio_step chunks of 64 sources it has summed (0:
// never), and starts at level prio0.
constexpr uint32_t kPrioStepSingle = 64;
// A single-system group starts at level (chunks it summed last step) /
// kPrioCarry; the batched force launch does the same per work item.
constexpr uint32_t kPrioCarry = 24;

__device__ __forceinline__ void set_issue_priority(uint32_t level) {
    if (level >= 3) __builtin_amdgcn_s_setprio(3);
    else if (level == 2) __builtin_amdgcn_s_setprio(2);
    else if (level == 1) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
}

struct WalkTree {
    const float4 *__restrict__ node4;
    const uint4 *__restrict__ child;
    uint32_t root, end;  // first node slot, one past the last
    uint32_t n_in;       // particles in the tree
};

// Walks one group for R * 8 of its W targets, t = part * 8 R + slot * R + r of
// the group.  px, py: the group's particle lane & (W - 1), or any real one of
// the group in place of one that is not; nreal: its real particles.  Returns in lane l the acceleration of
// target part * 8 R + l / (8 / R); vis and acc grow by the group's real-lane
// visits and acceptances, chunks becomes the sources summed / 64.
template <int W, int R, bool kWide>
__device__ __forceinline__ void walk_group(const WalkTree &tree, WalkShared &sh, uint32_t part,
                                           float px, float py, uint32_t nreal, float eps2, float theta2, uint32_t prio_step,
                                           uint32_t prio0, float &ax_out, float &ay_out,
                                           unsigned long long &vis, unsigned long long &acc,
                                           uint32_t &chunks) {
    const uint32_t lane = threadIdx.x & 63, stream = lane & 7u;
    uint32_t *const stack = sh.stack;
    uint32_t *const list = reinterpret_cast<uint32_t *>(sh.list4);
    float tx[R], ty[R], ax[R], ay[R];
    float vx[W / 8], vy[W / 8];  // this slot's share of the group, for the votes
    BoxXY box;
    {
        // the group through LDS: the targets are R consecutive particles a slot
        float2 *const xy = reinterpret_cast<float2 *>(stack);
        xy[lane] = make_float2(px, py);
        wave_lds_order();
        const uint32_t t0 = part * (8 * R) + (lane >> 3) * R, v0 = (lane >> 3) * (W / 8);
#pragma unroll
        for (int i = 0; i < W / 8; ++i) {
            const float2 p = xy[v0 + i];
            vx[i] = p.x;
            vy[i] = p.y;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float2 p = xy[t0 + r];
            tx[r] = p.x;
            ty[r] = p.y;
            ax[r] = 0.0f;
            ay[r] = 0.0f;
        }
        wave_lds_order();
        box.x0 = wave_extreme<false>(px);
        box.x1 = wave_extreme<true>(px);
        box.y0 = wave_extreme<false>(py);
        box.y1 = wave_extreme<true>(py);
    }
    float ev = eps2;  // in a vector register: a scalar operand costs the second issue
    asm volatile("" : "+v"(ev));
    uint32_t sp = 0, sc = 0, sources = 0;
    uint32_t visited = 0, accepted = 0;  // nodes, of this group
    if (nreal && tree.n_in) {            // one particle alone has no cell above it
        if (tree.n_in > 1u) {
            stack[lane] = tree.root;
            sp = 1;
        } else {
            list[lane] = source_key<kWide>(tree.root);
            sc = visited = accepted = 1;
        }
        wave_lds_order();
    }
    uint32_t level = prio_step ? min(prio0, 3u) : 0u;
    if (level) set_issue_priority(level);
    unsigned long long runs = 0;  // lanes whose opened leaf cell is not yet listed
    uint32_t run_first = 0, run_left = 0;
    uint32_t slot = 0, count = 0;
    while (true) {
        while (sc <= kWalkList - 64u && (run_left || runs || sp)) {
            if (run_left || runs) {
                if (!run_left) {
                    const uint32_t j = (uint32_t)__builtin_ctzll(runs);
                    runs &= runs - 1;
                    run_first = (uint32_t)__builtin_amdgcn_readlane(slot, j) + 1u;
                    run_left = min((uint32_t)__builtin_amdgcn_readlane(count, j),
                                   tree.end - min(run_first, tree.end));
                    visited += run_left;
                    accepted += run_left;
                }
                const uint32_t take = min(run_left, 64u);
                // entries past `take` are overwritten by the next append
                list[sc + lane] = source_key<kWide>(run_first + lane);
                sc += take;
                run_first += take;
                run_left -= take;
                continue;
            }
            // visit the top n cells of the stack (at least four entries stay
            // free, whatever the tree)
            sp = min(sp, kWalkStack - 4u);
            const uint32_t room = kWalkStack - kWalkMargin;
            uint32_t n = min(sp, 64u);
            if (sp + 3u * n > room) n = max(1u, (room - min(sp, room)) / 3u);
            n = uniform(n);
            sp -= n;
            const unsigned long long on = ~0ull >> (64u - n);
            wave_lds_order();
            slot = min(stack[sp + lane], tree.end - 1u);  // lanes past n: any node
            wave_lds_order();
            const float4 nd = tree_record<kWide>(tree.node4, slot);
            const uint4 ch = tree_record<kWide>(tree.child, slot);
            // ForceShader.comp:124-125 at the nearest point of the box
            const float nx = nd.x - __builtin_amdgcn_fmed3f(nd.x, box.x0, box.x1);
            const float ny = nd.y - __builtin_amdgcn_fmed3f(nd.y, box.y0, box.y1);
            const float near2 = (nx * nx + ny * ny) + eps2;
            // a particle's node has radius 0
            unsigned long long take = (__builtin_amdgcn_ballot_w64(nd.w <= 0.0f) |
                                       __builtin_amdgcn_ballot_w64(nd.w <= near2 * theta2)) &
                                      on;
            // the others eight at a time: this lane's stream names the cell,
            // its slot W / 8 of the particles.  Rounding is monotonic, so the
            // particle with the smallest dx*dx + dy*dy decides for them all.
            const unsigned long long vote = on & ~take;
            if (vote) {
                const uint32_t rank = lane_rank(vote), voted = (uint32_t)__popcll(vote);
                if (__builtin_amdgcn_inverse_ballot_w64(vote)) sh.cell[rank] = nd;
                wave_lds_order();
                unsigned long long opened = 0;  // by rank
                for (uint32_t base = 0; base < voted; base += 8) {
                    const float4 c = sh.cell[base + stream];
                    float least = 0.0f;
#pragma unroll
                    for (int i = 0; i < W / 8; ++i) {
                        const float dx = c.x - vx[i], dy = c.y - vy[i];
                        const float d2 = dx * dx + dy * dy;
                        least = i ? fminf(least, d2) : d2;
                    }
                    unsigned long long m =
                        __builtin_amdgcn_ballot_w64(!(c.w <= (least + eps2) * theta2));
                    m |= m >> 32;  // over the slots
                    m |= m >> 16;
                    m |= m >> 8;
                    opened |= (m & 0xffull) << base;
                }
                take |= __builtin_amdgcn_ballot_w64(((opened >> rank) & 1ull) == 0ull) & vote;
            }
            visited += n;
            const uint32_t taken = (uint32_t)__popcll(take);
            accepted += taken;
            if (__builtin_amdgcn_inverse_ballot_w64(take))
                list[sc + lane_rank(take)] = source_key<kWide>(slot);
            sc += taken;
            const unsigned long long open = on & ~take;
            runs = __builtin_amdgcn_ballot_w64(ch.w == kLeafMark) & open;
            count = ch.x;
            // the children of the others, by quadrant
            const unsigned long long inner = open & ~runs;
            if (inner) {
                const uint32_t size[4] = {ch.x, ch.y, ch.z, ch.w};
                uint32_t at = slot + 1u;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const unsigned long long m = __builtin_amdgcn_ballot_w64(size[q] != 0u) & inner;
                    if (__builtin_amdgcn_inverse_ballot_w64(m)) stack[sp + lane_rank(m)] = at;
                    sp += (uint32_t)__popcll(m);
                    at += size[q];
                }
            }
        }
        wave_lds_order();
        const uint32_t blocks = sc >> 5;
        sources += sc & ~31u;
        if (prio_step) {  // this wave's walk so far, in chunks
            const uint32_t want = min((sources >> 6) / prio_step, 3u);
            if (want > level) {
                level = want;
                set_issue_priority(level);
            }
        }
        sum_blocks<R, kWide>(sh, blocks, stream, tree.node4, tx, ty, ev, ax, ay);
        const uint32_t rest = sc & 31u;
        if (!run_left && !runs && !sp) {
            sum_rest<R, kWide>(sh, sc - rest, rest, stream, tree.node4, tx, ty, ev, ax, ay);
            sources += rest;
            break;
        }
        wave_lds_order();
        const uint32_t keep = lane < rest ? list[sc - rest + lane] : 0u;
        wave_lds_order();
        if (lane < rest) list[lane] = keep;
        sc = rest;
    }
    if (level) __builtin_amdgcn_s_setprio(0);  // a persistent wave goes on to other work
    vis += (unsigned long long)visited * nreal;
    acc += (unsigned long long)accepted * nreal;
    chunks = (sources + 63u) >> 6;
    ax_out = sum_streams<R>(ax, lane);
    ay_out = sum_streams<R>(ay, lane);
}

}  // namespace gsim
