// window_tile.hpp — an order by window whose elements may come in any order
// inside a window: counts, prefixes and ranks shared by the window-ordered
// gather and scatter (gs_staged.hip) and the hash join (join.hip).
//
// Elements are cut into chunks of kStChunk, tiles of a few chunks and groups
// of tiles.  A kernel of the caller counts every chunk's elements per window,
// k_st_groups and k_st_totals sum the counts up, and a split writes each tile,
// ordered by window in LDS, to them: since the order inside a window is free,
// an element's rank is one LDS atomic with return.
#pragma once
#include <algorithm>
#include "device.hpp"
#include "split_tile.hpp"

namespace edpp {
namespace {

constexpr int kStMaxWindows = 1024;
constexpr int kStBlock = 512;              // lanes of the splits
constexpr uint32_t kStNone = 0xFFFFFFFFu;  // no element
constexpr int kStRowBlock = 1024;
constexpr int kStChunk = 4096;             // elements whose counts are kept together
constexpr int kStMaxGroup = 64;            // tiles of a group whose prefixes are kept together
constexpr int kStGates = 64, kStGatePad = 32;  // words, a 128-byte line each

// elements [v*E, v*E + E) of p; `none` for the ones at or past n
template <class T, int E>
__device__ __forceinline__ void st_load(const T* __restrict__ p, int64_t v, int64_t n, T none, T* x) {
    if (E * v + E <= n) {
        typedef T vec __attribute__((ext_vector_type(E)));
        const vec y = ld_stream(reinterpret_cast<const vec*>(p) + v);
        #pragma unroll
        for (int k = 0; k < E; ++k) x[k] = y[k];
    } else {
        #pragma unroll
        for (int k = 0; k < E; ++k) x[k] = E * v + k < n ? p[E * v + k] : none;
    }
}
// p[E*v + k] = x[k] where ok[k] (elements at or past n are never ok)
template <class T, int E>
__device__ __forceinline__ void st_store(T* __restrict__ p, int64_t v, const T* x, const bool* ok) {
    bool all = true;
    #pragma unroll
    for (int k = 0; k < E; ++k) all = all && ok[k];
    if (all) {
        typedef T vec __attribute__((ext_vector_type(E)));
        vec y;
        #pragma unroll
        for (int k = 0; k < E; ++k) y[k] = x[k];
        st_stream(y, reinterpret_cast<vec*>(p) + v);
    } else {
        #pragma unroll
        for (int k = 0; k < E; ++k)
            if (ok[k]) p[E * v + k] = x[k];
    }
}

struct StGeom {
    int64_t n;
    int shift;          // window of an index: idx >> shift
    int W;              // windows
    int WP;             // W, rounded up to even
    int64_t chunks, tiles, groups;
    int group;          // tiles per group, a power of two up to kStMaxGroup
    int xcds;
    uint32_t near;      // a gather's chunk whose indices span fewer elements is done directly
    uint32_t* probe;    // [2 * workgroup] distinct lines and elements that a gather's k_st_probe saw
    uint8_t* done;      // [chunks] chunk is finished (null: none is)
    uint16_t* count;    // [chunk][WP] elements per window of the chunks that are not
    uint32_t* rows;     // [tile][WP] elements of the window in the group's earlier tiles
    uint32_t* gsum;     // [group][WP] the group's elements, then those of the earlier groups
    uint32_t* total;    // [WP] elements of each window
    uint32_t* base;     // [W + 1] first position of each window; base[W] = elements staged
    // a second split: windows into bins
    int sub_shift;      // bin of an index: idx >> sub_shift
    int lg_subs;
    uint32_t* tile2;    // [W + 1] first second-level tile of each window
    uint16_t* win2;     // window of each second-level tile
    uint32_t* rows2;    // [window][bin][tile of the window]
    uint32_t* bins;     // [W << lg_subs] first position of each bin
    uint32_t* gate;     // [kStGates] some not 0: some chunk is not finished; 0 between calls (null: always so)
    uint32_t* open;     // whether gate was set, for the kernels behind k_st_groups (with a gate)
};
__device__ __forceinline__ uint32_t* st_gate(const StGeom& g, uint32_t i) {
    return g.gate + i % kStGates * kStGatePad;
}
// by the call's last kernel
__device__ __forceinline__ void st_close(const StGeom& g) {
    if (blockIdx.x == 0 && threadIdx.x < kStGates) *st_gate(g, threadIdx.x) = 0u;
}
// The o-th of `count` workgroups or steps in XCD order: contiguous ranges per
// XCD, as split_tile.hpp's xcd_tile, for the 8 XCDs of the chip
__device__ __forceinline__ uint32_t st_order(uint32_t o, uint32_t count, int xcds) {
    if (xcds == 8 && count >= 8) {
        const uint32_t per = count >> 3, rem = count & 7u, x = o & 7u;
        return x * per + std::min(x, rem) + (o >> 3);
    }
    return o;
}
// Counters per bucket: lanes that count the same bucket at once serialize, so
// few buckets get several counters each, taken by lane
__host__ __device__ constexpr int st_copies_lg(int B) { return B <= 64 ? 3 : B <= 128 ? 2 : B <= 256 ? 1 : 0; }

constexpr int kStBuckets = 1024 + 8;

// Exclusive prefix of cnt[0, C) into off[], C <= 2*kStBlock, two entries per
// lane; returns the sum.  A barrier before and after.
__device__ __forceinline__ uint32_t st_scan(uint32_t tid, const uint32_t* cnt, uint32_t* off, int C, uint32_t* wtmp) {
    const int t = (int)tid, w = __builtin_amdgcn_readfirstlane(t / kWave);
    __syncthreads();
    const uint32_t a = 2 * t < C ? cnt[2 * t] : 0u, b = 2 * t + 1 < C ? cnt[2 * t + 1] : 0u;
    const uint32_t inc = wave_inclusive_add(a + b);
    if (lane_id() == kWave - 1) wtmp[w] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
    #pragma unroll
    for (int q = 0; q < kStBlock / kWave; ++q) {
        before += q < w ? wtmp[q] : 0u;
        all += wtmp[q];
    }
    const uint32_t x = before + inc - a - b;
    if (2 * t < C) off[2 * t] = x;
    if (2 * t + 1 < C) off[2 * t + 1] = x + a;
    __syncthreads();
    return all;
}

// Slots of the lane's elements in bucket order, two per word of at[], from
// one counter atomic each (1 << cl counters per bucket, taken by lane);
// bucket(e, x[e]) is the e-th element's bucket, B for one that is none; off[b
// << cl] = first slot of bucket b.  Returns the number of elements that are
// some; the others all get the last slot, which is then past them.
template <int EPL, class Bucket>
__device__ __forceinline__ uint32_t st_rank(uint32_t tid, uint32_t (&x)[EPL], uint32_t (&at)[EPL / 2],
                                            const Bucket& bucket, int B, int cl, uint32_t* cnt, uint32_t* off,
                                            uint32_t* wtmp) {
    for (int i = (int)tid; i < ((B + 1) << cl); i += kStBlock) cnt[i] = 0;
    __syncthreads();
    const uint32_t copy = tid & ((1u << cl) - 1u);
    #pragma unroll
    for (int e = 0; e < EPL / 2; ++e) {
        const uint32_t r0 = __hip_atomic_fetch_add(cnt + (bucket(2 * e, x[2 * e]) << cl) + copy,
                                                   1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const uint32_t r1 = __hip_atomic_fetch_add(cnt + (bucket(2 * e + 1, x[2 * e + 1]) << cl) + copy,
                                                   1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        at[e] = r0 | (r1 << 16);
    }
    // Packed before the scan, and the buckets worked out again after it: held
    // across it, ranks and counter addresses do not fit the registers of two
    // workgroups per CU.
    #pragma unroll
    for (int e = 0; e < EPL / 2; ++e) asm volatile("" : "+v"(at[e]), "+v"(x[2 * e]), "+v"(x[2 * e + 1]));
    constexpr uint32_t kLast = kStBlock * EPL - 1;
    if (tid < (1u << cl)) off[(B << cl) + tid] = kLast;
    const uint32_t m = st_scan(tid, cnt, off, B << cl, wtmp);
    #pragma unroll
    for (int e = 0; e < EPL / 2; ++e) {
        const uint32_t o0 = off[(bucket(2 * e, x[2 * e]) << cl) + copy];
        const uint32_t o1 = off[(bucket(2 * e + 1, x[2 * e + 1]) << cl) + copy];
        at[e] = std::min((at[e] & 0xFFFFu) + o0, kLast) | std::min((at[e] >> 16) + o1, kLast) << 16;
    }
    return m;
}
// v[e] to slot e's place in buf
template <class V, int EPL>
__device__ __forceinline__ void st_place(V* buf, const uint32_t (&at)[EPL / 2], const V (&v)[EPL]) {
    #pragma unroll
    for (int e = 0; e < EPL / 2; ++e) {
        buf[at[e] & 0xFFFFu] = v[2 * e];
        buf[at[e] >> 16] = v[2 * e + 1];
    }
}
// Prefixes of the windows' counts, in three steps of which each takes a launch
// (or is part of the split) and none hands data from one workgroup to another:
// the release and acquire that such a step in one kernel takes write back and
// invalidate whole L2s (2 x 2^24 keys in 1024 windows: 72 us in one kernel,
// 80 with a single workgroup for the last step).
//
// k_st_groups: workgroup = one group of g.group tiles and one slice of the
// windows (grid.z), cut into parts of tiles, one lane for two windows of a
// part: rows[] within the group, gsum[] the group's sums.  grid.y = 2 takes
// two problems in one launch.
template <int CH>
__global__ __launch_bounds__(kStRowBlock) void k_st_groups(StGeom g0, StGeom g1, int lgp) {
    const StGeom& g = blockIdx.y ? g1 : g0;
    if ((int64_t)blockIdx.x >= g.groups) return;
    __shared__ uint32_t part[2 * kStRowBlock];
    __shared__ uint8_t fin[kStMaxGroup * CH];
    const int x = threadIdx.x;
    const int l = x & ((1 << lgp) - 1), q = x >> lgp;  // pair of windows in the slice, part
    const int np = kStRowBlock >> lgp;                 // parts, at most g.group
    const int per = g.group / np;
    const int P = g.WP / 2;
    const int p = ((int)blockIdx.z << lgp) + l;        // windows 2p and 2p + 1
    const bool in = p < P;
    const int64_t t0 = (int64_t)blockIdx.x * g.group;
    if (g.gate) {
        const bool open = ballot(*st_gate(g, lane_id()) != 0) != 0;  // the same in every wave
        if (blockIdx.x == 0 && blockIdx.z == 0 && x == 0) *g.open = open ? 1u : 0u;
        if (!open) return;
    }
    for (int i = x; i < g.group * CH; i += kStRowBlock)
        fin[i] = t0 * CH + i >= g.chunks || (g.done && g.done[t0 * CH + i]) ? 1 : 0;
    __syncthreads();
    const uint32_t* cnt = reinterpret_cast<const uint32_t*>(g.count) + p;
    auto tile = [&](int t, uint32_t& u, uint32_t& v) {  // the counts of one tile; finished chunks have none
        #pragma unroll
        for (int k = 0; k < CH; ++k) {
            const int64_t c = std::min<int64_t>((t0 + t) * CH + k, g.chunks - 1);
            const uint32_t y = cnt[c * P];
            const bool f = fin[t * CH + k] != 0;
            u += f ? 0u : y & 0xFFFFu;
            v += f ? 0u : y >> 16;
        }
    };
    uint32_t a = 0, b = 0;
    if (in) {
        #pragma unroll 4
        for (int t = q * per; t < (q + 1) * per; ++t) tile(t, a, b);
    }
    part[2 * x] = a;
    part[2 * x + 1] = b;
    __syncthreads();
    a = b = 0;
    for (int k = 0; k < q; ++k) {
        a += part[2 * ((k << lgp) + l)];
        b += part[2 * ((k << lgp) + l) + 1];
    }
    if (in) {
        uint2* rows = reinterpret_cast<uint2*>(g.rows) + p;
        #pragma unroll 4
        for (int t = q * per; t < (q + 1) * per; ++t) {
            if (t0 + t < g.tiles) rows[(t0 + t) * P] = make_uint2(a, b);
            tile(t, a, b);
        }
        if (q == np - 1) reinterpret_cast<uint2*>(g.gsum)[(int64_t)blockIdx.x * P + p] = make_uint2(a, b);
    }
}
// k_st_totals: workgroup = one slice of the windows; gsum[] becomes the
// elements of the earlier groups, total[] those of the window
template <int CH>
__global__ __launch_bounds__(kStRowBlock) void k_st_totals(StGeom g0, StGeom g1, int lgp) {
    const StGeom& g = blockIdx.y ? g1 : g0;
    __shared__ uint32_t part[2 * kStRowBlock];
    if (g.gate && *g.open == 0) return;
    const int x = threadIdx.x;
    const int l = x & ((1 << lgp) - 1), q = x >> lgp;
    const int np = kStRowBlock >> lgp;
    const int P = g.WP / 2;
    const int p = ((int)blockIdx.x << lgp) + l;
    const bool in = p < P;
    uint2* gsum = reinterpret_cast<uint2*>(g.gsum) + p;
    const int64_t gper = (g.groups + np - 1) / np;
    const int64_t k0 = std::min<int64_t>(q * gper, g.groups), k1 = std::min<int64_t>(k0 + gper, g.groups);
    uint32_t a = 0, b = 0;
    if (in) {
        #pragma unroll 16
        for (int64_t k = k0; k < k1; ++k) {
            const uint2 y = gsum[k * P];
            a += y.x;
            b += y.y;
        }
    }
    part[2 * x] = a;
    part[2 * x + 1] = b;
    __syncthreads();
    uint32_t ta = 0, tb = 0;
    a = b = 0;
    for (int k = 0; k < np; ++k) {
        const uint32_t ya = part[2 * ((k << lgp) + l)], yb = part[2 * ((k << lgp) + l) + 1];
        a += k < q ? ya : 0u;
        b += k < q ? yb : 0u;
        ta += ya;
        tb += yb;
    }
    if (in) {
        #pragma unroll 16
        for (int64_t k = k0; k < k1; ++k) {
            const uint2 y = gsum[k * P];
            gsum[k * P] = make_uint2(a, b);
            a += y.x;
            b += y.y;
        }
        if (q == 0) reinterpret_cast<uint2*>(g.total)[p] = make_uint2(ta, tb);
    }
}
// First positions of the lane's windows 2*tid and 2*tid + 1 from total[], in
// every workgroup of a split (kStBlock lanes, at most 2*kStBlock windows).  A
// barrier inside.
__device__ __forceinline__ uint2 st_bases(const StGeom& g, uint32_t tid, uint32_t* wtmp) {
    const bool in = (int)tid < g.WP / 2;
    const uint2 y = in ? reinterpret_cast<const uint2*>(g.total)[tid] : make_uint2(0, 0);
    const int w = __builtin_amdgcn_readfirstlane((int)tid / kWave);
    const uint32_t inc = wave_inclusive_add(y.x + y.y);
    if (lane_id() == kWave - 1) wtmp[w] = inc;
    __syncthreads();
    uint32_t before = 0;
    #pragma unroll
    for (int q = 0; q < kStBlock / kWave; ++q) before += q < w ? wtmp[q] : 0u;
    const uint32_t first = before + inc - y.x - y.y;
    return make_uint2(first, first + y.x);
}
// The split's first workgroup keeps the bases (and a second split's tiles of
// CH chunks) for the kernels behind it.  t2s: kStMaxWindows words of LDS.
template <int CH>
__device__ __forceinline__ void st_keep_bases(const StGeom& g, uint32_t tid, uint32_t* wtmp, uint32_t* t2s) {
    const uint2 f = st_bases(g, tid, wtmp);
    const bool in = (int)tid < g.WP / 2;
    const uint2 y = in ? reinterpret_cast<const uint2*>(g.total)[tid] : make_uint2(0, 0);
    if (in) {  // base[] and tile2[] have room for WP + 1
        g.base[2 * tid] = f.x;
        g.base[2 * tid + 1] = f.y;
    }
    __syncthreads();
    if ((int)tid == g.WP / 2 - 1) g.base[g.W] = f.y + (g.W == g.WP ? y.y : 0u);  // an odd W's last pair has one window
    if (!g.tile2) return;
    constexpr uint32_t kTile = CH * kStChunk;
    const uint32_t na = (y.x + kTile - 1) / kTile, nb = (y.y + kTile - 1) / kTile;
    const int w = __builtin_amdgcn_readfirstlane((int)tid / kWave);
    const uint32_t inc = wave_inclusive_add(na + nb);
    if (lane_id() == kWave - 1) wtmp[w] = inc;
    __syncthreads();
    uint32_t before = 0, tiles2 = 0;
    #pragma unroll
    for (int q = 0; q < kStBlock / kWave; ++q) {
        before += q < w ? wtmp[q] : 0u;
        tiles2 += wtmp[q];
    }
    const uint32_t t2 = before + inc - na - nb;
    if (in) {
        g.tile2[2 * tid] = t2s[2 * tid] = t2;
        g.tile2[2 * tid + 1] = t2s[2 * tid + 1] = t2 + na;
    }
    __syncthreads();
    if (tid == 0) g.tile2[g.W] = tiles2;
    for (uint32_t t = tid; t < tiles2; t += kStBlock) {
        int lo = 0, hi = g.W;  // last window whose first tile is at or before t: empty windows have none
        while (hi - lo > 1) {
            const int m = (lo + hi) / 2;
            if (t2s[m] <= t) lo = m;
            else hi = m;
        }
        g.win2[t] = (uint16_t)lo;
    }
    __syncthreads();
}
// cnt[w] = distance from a slot of the tile to its output position, once the
// tile's slots are ranked (off[w << cl] the window's first one)
__device__ __forceinline__ void st_distances(const StGeom& g, int64_t tile, uint32_t tid, int cl, uint32_t* cnt,
                                             const uint32_t* off, uint32_t* wtmp) {
    const uint2 f = st_bases(g, tid, wtmp);
    if ((int)tid < g.WP / 2) {
        const uint2 gs = reinterpret_cast<const uint2*>(g.gsum + tile / g.group * g.WP)[tid];
        const uint2 rw = reinterpret_cast<const uint2*>(g.rows + tile * g.WP)[tid];
        cnt[2 * tid] = f.x + gs.x + rw.x - off[(2 * tid) << cl];
        cnt[2 * tid + 1] = f.y + gs.y + rw.y - off[(2 * tid + 1) << cl];
    }
}

// Host side: tiles per group (up to some 256 groups, each a workgroup of
// k_st_groups or one per slice); the launches for one problem or two of the
// same window count and group size.
inline int st_group(int64_t tiles) {
    int g = 8;
    while (g < kStMaxGroup && tiles / g > 256) g *= 2;
    return g;
}
template <int CH>
inline void launch_st_prefix(hipStream_t stream, const StGeom& g0, const StGeom* g1) {
    int l = 0;  // log2 of a slice's pairs of windows: at most one part per tile, 128 pairs where there are as many
    while ((kStRowBlock >> l) > g0.group || (l < 7 && (2 << l) < g0.WP)) ++l;
    const int64_t groups = g1 ? std::max(g0.groups, g1->groups) : g0.groups;
    const unsigned slices = (unsigned)((g0.WP / 2 + (1 << l) - 1) >> l), two = g1 ? 2 : 1;
    const StGeom& ga = g0;
    const StGeom& gb = g1 ? *g1 : g0;
    hipLaunchKernelGGL((k_st_groups<CH>), dim3((unsigned)groups, two, slices), dim3(kStRowBlock), 0, stream, ga, gb, l);
    hipLaunchKernelGGL((k_st_totals<CH>), dim3(slices, two), dim3(kStRowBlock), 0, stream, ga, gb, l);
}

}  // namespace
}  // namespace edpp
