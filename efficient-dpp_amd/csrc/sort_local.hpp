// sort_local.hpp — the end of a long radix sort: keys in order of their top
// bits become fully ordered, one segment of equal top bits at a time, in LDS.
//
// The top 16 bits take two stable split passes; the low 16 would take two
// more, of which each reads the keys twice and writes 256 runs per tile.  In
// their place a workgroup reads each segment once, ranks it twice in LDS and
// writes it once, in place.  That needs short segments: k_sort_sample and
// k_sort_decide look at 2^14 keys, and where the top bits are far from evenly
// spread (gate), the two splits run instead.  A segment that does not fit all
// the same goes to a list: k_sort_long orders it in LDS up to 4992 keys,
// k_sort_longer through the spare copies beyond.
//
// 2^28 even pairs, in us: k_sort_local 1030 to 1070 in place of 2 x 1240 for
// two passes, the others and the passes that leave at once about 110 (starts
// 23, scans of unused counts 35); the sort 4900 before, 3650 now, of keys alone
// 3890 and 2900.  k_sort_local moves 4.3 GB, 735 us of copying; 16 ballots and
// two rounds through LDS hold the vector units for 135 cycles of a CU per 64
// pairs, 110 of the LDS.  Slower: 1024 lanes and segments of 8192 (1870), hist
// in 32 bits (three workgroups per CU instead of four, 1160), several segments
// per workgroup (1300), the compiler's own form of the match (keys alone 980
// instead of 830).  Keys far from even pay for the look and the launches
// that leave: 38 us at 2^26, 54 at 2^28, which is 4790 instead of 4740 (2^28
// pairs of 20 bits) and 3 to 4 % at 2^26.  The look lets a segment pass that
// holds up to 0.1 % of the keys: one such segment, which a single workgroup
// then orders, takes the gain (2^26 pairs 1310 instead of 1280, 2^28 5000
// instead of 4960), three of half the size leave most of it (1210, 4320).
#pragma once
#include <algorithm>
#include "ctx.hpp"
#include "device.hpp"
#include "split_tile.hpp"

namespace edpp {
namespace {

constexpr int kSlBlock = 512;
constexpr int kSlRows = 9, kSlCap = 69 * kWave;          // k_sort_local: four workgroups' LDS per CU
constexpr int kSlLongRows = 10, kSlLongCap = 78 * kWave;  // k_sort_long: three
constexpr int kSlIdxBits = 13;
constexpr int kSlSamples = 1 << 14;
constexpr int kSlHot = 16;  // a segment of this many samples is too long for one workgroup
static_assert(kSlCap <= kSlRows * kSlBlock && kSlLongCap <= kSlLongRows * kSlBlock && kSlLongCap <= 1 << kSlIdxBits);

struct SlGeom {
    int64_t n;
    int segs;         // 1 << top bits
    uint32_t flip;    // 0, or the sign bit
    uint16_t* sample; // [kSlSamples] top 16 bits
    uint32_t* start;  // [segs + 1] first key of each segment
    uint32_t* list;   // segments that do not fit k_sort_local
    uint32_t* gate;   // [0]: not 0: the segments are not short, split instead; [1]: entries of the list
};

__global__ __launch_bounds__(1024) void k_sort_sample(const uint32_t* __restrict__ keys, SlGeom g) {
    const uint32_t i = blockIdx.x * 1024u + threadIdx.x;
    g.sample[i] = (uint16_t)(keys[((uint64_t)mix32(i) * (uint64_t)g.n) >> 32] >> 16);
}

// Pairs of samples in one segment: even segments give about (samples)^2 / 2 /
// segs, 2048 to 8192; 1.15 times as many, and k_sort_long still takes most.
__global__ __launch_bounds__(1024) void k_sort_decide(SlGeom g) {
    extern __shared__ uint32_t cnt[];  // [segs] 16-bit counts
    __shared__ uint32_t pairs, most;
    uint32_t b[kSlSamples / 1024];
    #pragma unroll
    for (int i = 0; i < kSlSamples / 1024; ++i) b[i] = g.sample[i * 1024 + threadIdx.x];
    for (int i = threadIdx.x; i < g.segs / 2; i += 1024) cnt[i] = 0;
    if (threadIdx.x == 0) pairs = most = 0;
    __syncthreads();
    uint32_t p = 0;
    bool hot = false;
    #pragma unroll
    for (int i = 0; i < kSlSamples / 1024; ++i) {
        const uint32_t s = b[i] / (65536u / (uint32_t)g.segs), sh = (s & 1u) * 16u;
        const uint32_t old = (__hip_atomic_fetch_add(cnt + (s >> 1), 1u << sh, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_WORKGROUP) >> sh) & 0xFFFFu;
        p += old;
        hot = hot || old >= kSlHot;
    }
    p = wave_sum(p);
    if (lane_id() == 0) __hip_atomic_fetch_add(&pairs, p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    hot = __syncthreads_or(hot);
    if (threadIdx.x == 0) {
        const uint32_t even = (uint32_t)kSlSamples * (uint32_t)kSlSamples / 2 / (uint32_t)g.segs;
        g.gate[0] = hot || pairs > even / 20 * 23 ? 1u : 0u;
        g.gate[1] = 0u;
    }
}

// start[s] = the first key whose top bits are s or more, from where it would
// be if the segments were even, in steps that double
__global__ __launch_bounds__(256) void k_sort_starts(const uint32_t* __restrict__ keys, SlGeom g) {
    if (g.gate[0]) return;
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s > g.segs) return;
    int64_t lo = 0, hi = g.n;  // keys before lo are less, keys from hi on are not
    if (s > 0 && s < g.segs) {
        const uint32_t first = (uint32_t)((uint64_t)s * (0x100000000ull / (uint64_t)g.segs));
        auto less = [&](int64_t i) { return (keys[i] ^ g.flip) < first; };
        int64_t at = (int64_t)((uint64_t)s * (uint64_t)g.n / (uint64_t)g.segs);
        const bool up = less(at);
        for (int64_t step = 4096; lo < hi; step *= 2) {
            if (up) {
                lo = at + 1;
                at += step;
                if (at >= hi) break;
                if (!less(at)) {
                    hi = at;
                    break;
                }
            } else {
                hi = at;
                at -= step;
                if (at < lo) break;
                if (less(at)) {
                    lo = at + 1;
                    break;
                }
            }
        }
        while (lo < hi) {
            const int64_t mid = lo + (hi - lo) / 2;
            if (less(mid)) lo = mid + 1;
            else hi = mid;
        }
    } else if (s > 0) {
        lo = g.n;
    }
    g.start[s] = (uint32_t)lo;
}

// Stable ranks of the wave's rows among its own elements, old[j] + below[j] of
// a lane's item j < rows, and its counts per digit in row[], which are cleared
// by pairs (each row starts on a word) before they are counted.
typedef uint32_t __attribute__((may_alias)) SlPair;
template <int BITS, int SHIFT, int ROWS>
__device__ __forceinline__ void sl_rank(const uint32_t (&x)[ROWS], int rows, uint16_t* row, uint32_t (&old)[ROWS],
                                        uint32_t (&below)[ROWS]) {
    constexpr int B = 1 << BITS;
    #pragma unroll
    for (int i = 0; i < B / kWave / 2; ++i) reinterpret_cast<SlPair*>(row)[i * kWave + lane_id()] = 0;
    #pragma unroll
    for (int j = 0; j < ROWS; ++j) {
        if (j >= rows) continue;
        uint32_t lo = ~0u, hi = ~0u;
        #pragma unroll
        for (int bit = 0; bit < BITS; ++bit) {
            // lo & ~(bal ^ on) in one instruction: the compiler's own form takes a third more
            const uint32_t on = (uint32_t)__builtin_amdgcn_sbfe((int)x[j], SHIFT + bit, 1);
            const uint64_t bal = ballot((int)on < 0);
            lo = __builtin_amdgcn_bitop3_b32(lo, (uint32_t)bal, on, 0x90);
            hi = __builtin_amdgcn_bitop3_b32(hi, (uint32_t)(bal >> 32), on, 0x90);
        }
        below[j] = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
        // the wave's LDS operations run in order: its earlier rows, then this one
        uint16_t* at = row + __builtin_amdgcn_ubfe(x[j], SHIFT, BITS);
        old[j] = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        if (below[j] == 0)
            __hip_atomic_store(at, (uint16_t)(old[j] + __popc(lo) + __popc(hi)), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
}

// Exclusive prefix of every lane's x over the workgroup's first WAVES waves;
// one barrier.
template <int WAVES>
__device__ __forceinline__ uint32_t sl_prefix(uint32_t x, uint32_t* wtmp) {
    const int w = threadIdx.x / kWave;
    const uint32_t inc = wave_inclusive_add(x);
    if (lane_id() == kWave - 1) wtmp[w] = inc;
    __syncthreads();
    uint32_t at = inc - x;
    #pragma unroll
    for (int q = 0; q < WAVES; ++q) at += q < w ? wtmp[q] : 0u;
    return at;
}

// hist[w][b] = elements of smaller digits, and of digit b in earlier waves.
// Barriers around it.
template <int BITS, int BLOCK = kSlBlock>
__device__ __forceinline__ void sl_scan(uint16_t* hist, uint32_t* wtmp) {
    constexpr int B = 1 << BITS, W = BLOCK / kWave;
    static_assert(B <= BLOCK);
    const int t = threadIdx.x;
    __syncthreads();
    uint32_t c[W], sum = 0;
    if (t < B) {
        #pragma unroll
        for (int q = 0; q < W; ++q) c[q] = hist[q * B + t];
        #pragma unroll
        for (int q = 0; q < W; ++q) sum += c[q];
    }
    uint32_t at = sl_prefix<B / kWave>(sum, wtmp);
    if (t < B) {
        #pragma unroll
        for (int q = 0; q < W; ++q) {
            hist[q * B + t] = (uint16_t)at;
            at += c[q];
        }
    }
    __syncthreads();
}

// LDS of a workgroup that orders up to CAP keys
template <int CAP, bool KV, int BITS>
struct SlLds {
    uint32_t comp[CAP];
    int32_t val[KV ? CAP : 1];
    alignas(16) uint16_t hist[(kSlBlock / kWave) << BITS];
    uint32_t wtmp[kSlBlock / kWave];
};

// Orders the cnt <= CAP keys from s on, which agree above their low BITS1 +
// BITS2 bits (top), in place.  An element goes through LDS as one word, its
// low bits over its index; the value follows the index at the end.
template <int ROWS, bool KV, int BITS1, int BITS2, class Lds>
__device__ __forceinline__ void sl_segment(uint32_t* __restrict__ keys, int32_t* __restrict__ vals, uint32_t s, int cnt,
                                           uint32_t top, Lds& l) {
    constexpr int W = kSlBlock / kWave, SH = KV ? kSlIdxBits : 0;
    static_assert(SH + BITS1 + BITS2 <= 32 && BITS2 <= BITS1);
    // rows of 64 elements, dealt to the waves in order
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int all = (cnt + kWave - 1) / kWave, per = all / W, rem = all % W;
    const int rows = per + (w < rem ? 1 : 0);
    const int e0 = (w * per + std::min(w, rem)) * kWave + lane_id();
    uint32_t x[ROWS], old[ROWS], below[ROWS];
    const __amdgpu_buffer_rsrc_t kr = buf_rsrc(keys + s, cnt);
    #pragma unroll
    for (int j = 0; j < ROWS; ++j) x[j] = j < rows ? buf_load<uint32_t>(kr, (uint32_t)e0 * 4u, j * kWave * 4) : 0u;
    int32_t v[ROWS];
    if constexpr (KV) {
        const __amdgpu_buffer_rsrc_t vr = buf_rsrc(vals + s, cnt);
        #pragma unroll
        for (int j = 0; j < ROWS; ++j) v[j] = j < rows ? buf_load<int32_t>(vr, (uint32_t)e0 * 4u, j * kWave * 4) : 0;
    }
    // the last row's lanes past the end hold all ones: they stay the last ones
    #pragma unroll
    for (int j = 0; j < ROWS; ++j) {
        const uint32_t y = __builtin_amdgcn_ubfe(x[j], 0, BITS1 + BITS2);
        x[j] = e0 + j * kWave < cnt ? KV ? (y << SH) | (uint32_t)(e0 + j * kWave) : y : ~0u;
    }
    uint16_t* row = l.hist + (w << BITS1);
    sl_rank<BITS1, SH, ROWS>(x, rows, row, old, below);
    if constexpr (KV) {  // the values were on their way until here
        #pragma unroll
        for (int j = 0; j < ROWS; ++j)
            if (j < rows) l.val[e0 + j * kWave] = v[j];
    }
    sl_scan<BITS1>(l.hist, l.wtmp);
    #pragma unroll
    for (int j = 0; j < ROWS; ++j)
        if (j < rows) l.comp[row[__builtin_amdgcn_ubfe(x[j], SH, BITS1)] + old[j] + below[j]] = x[j];
    __syncthreads();
    #pragma unroll
    for (int j = 0; j < ROWS; ++j)
        if (j < rows) x[j] = l.comp[e0 + j * kWave];
    row = l.hist + (w << BITS2);
    sl_rank<BITS2, SH + BITS1, ROWS>(x, rows, row, old, below);
    sl_scan<BITS2>(l.hist, l.wtmp);
    #pragma unroll
    for (int j = 0; j < ROWS; ++j)
        if (j < rows) l.comp[row[__builtin_amdgcn_ubfe(x[j], SH + BITS1, BITS2)] + old[j] + below[j]] = x[j];
    __syncthreads();
    #pragma unroll
    for (int j = 0; j < ROWS; ++j) {
        const int e = j * kSlBlock + (int)threadIdx.x;
        if (e < cnt) {
            const uint32_t y = l.comp[e];
            keys[s + e] = top | __builtin_amdgcn_ubfe(y, SH, BITS1 + BITS2);
            if constexpr (KV) vals[s + e] = l.val[__builtin_amdgcn_ubfe(y, 0, SH)];
        }
    }
}

template <bool KV, int BITS1, int BITS2>
__global__ __launch_bounds__(kSlBlock) void k_sort_local(uint32_t* __restrict__ keys, int32_t* __restrict__ vals, SlGeom g) {
    __shared__ SlLds<kSlCap, KV, BITS1> l;
    if (g.gate[0]) return;
    const uint32_t s = g.start[blockIdx.x], cnt = g.start[blockIdx.x + 1] - s;
    if (cnt <= kSlCap) {
        if (cnt > 1)
            sl_segment<kSlRows, KV, BITS1, BITS2>(keys, vals, s, (int)cnt, (blockIdx.x << (BITS1 + BITS2)) ^ g.flip, l);
    } else if (threadIdx.x == 0) {
        g.list[__hip_atomic_fetch_add(g.gate + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)] = blockIdx.x;
    }
}

template <bool KV, int BITS1, int BITS2>
__global__ __launch_bounds__(kSlBlock) void k_sort_long(uint32_t* __restrict__ keys, int32_t* __restrict__ vals, SlGeom g) {
    __shared__ SlLds<kSlLongCap, KV, BITS1> l;
    if (g.gate[0]) return;
    const uint32_t entries = g.gate[1];
    for (uint32_t i = blockIdx.x; i < entries; i += gridDim.x) {
        const uint32_t seg = g.list[i], s = g.start[seg], cnt = g.start[seg + 1] - s;
        if (cnt > kSlLongCap) continue;
        sl_segment<kSlLongRows, KV, BITS1, BITS2>(keys, vals, s, (int)cnt, (seg << (BITS1 + BITS2)) ^ g.flip, l);
        __syncthreads();
    }
}

// One stable split of a long segment's keys [0, cnt) by BITS bits, by one workgroup
template <bool KV, int BITS, int SHIFT>
__device__ __forceinline__ void sl_long_pass(const uint32_t* ks, const int32_t* vs, uint32_t* kd, int32_t* vd,
                                             uint32_t cnt, uint16_t* hist, uint32_t* run, uint32_t* wtmp) {
    constexpr int B = 1 << BITS, R = 8, TILE = R * kSlBlock;
    const int t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t / kWave);
    if (t < B) run[t] = 0;
    __syncthreads();
    for (uint32_t e = t; e < cnt; e += kSlBlock)
        __hip_atomic_fetch_add(run + __builtin_amdgcn_ubfe(ks[e], SHIFT, BITS), 1u, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    const uint32_t first = sl_prefix<B / kWave>(t < B ? run[t] : 0u, wtmp);
    if (t < B) run[t] = first;
    for (uint32_t at = 0; at < cnt; at += TILE) {
        const uint32_t e0 = at + (uint32_t)(w * R * kWave) + lane_id();
        uint32_t x[R], old[R], below[R];
        int32_t v[R];
        #pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint32_t e = e0 + j * kWave;
            x[j] = e < cnt ? ks[e] : ~0u;  // past the end: the last ones
            if constexpr (KV) v[j] = e < cnt ? vs[e] : 0;
        }
        uint16_t* row = hist + (w << BITS);
        sl_rank<BITS, SHIFT, R>(x, R, row, old, below);
        sl_scan<BITS>(hist, wtmp);
        #pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint32_t d = __builtin_amdgcn_ubfe(x[j], SHIFT, BITS);
            const uint32_t p = run[d] + row[d] + old[j] + below[j] - hist[d];
            if (e0 + j * kWave < cnt) {
                kd[p] = x[j];
                if constexpr (KV) vd[p] = v[j];
            }
        }
        __syncthreads();
        if (t < B) run[t] += (t + 1 < B ? (uint32_t)hist[t + 1] : (uint32_t)TILE) - hist[t];
        __syncthreads();
    }
}

template <bool KV, int BITS1, int BITS2>
__global__ __launch_bounds__(kSlBlock) void k_sort_longer(uint32_t* keys, int32_t* vals, uint32_t* tkeys, int32_t* tvals,
                                                          SlGeom g) {
    __shared__ alignas(16) uint16_t hist[(kSlBlock / kWave) << BITS1];
    __shared__ uint32_t run[1 << BITS1], wtmp[kSlBlock / kWave];
    if (g.gate[0]) return;
    const uint32_t entries = g.gate[1];
    for (uint32_t i = blockIdx.x; i < entries; i += gridDim.x) {
        const uint32_t seg = g.list[i], s = g.start[seg], cnt = g.start[seg + 1] - s;
        if (cnt <= kSlLongCap) continue;
        sl_long_pass<KV, BITS1, 0>(keys + s, vals + s, tkeys + s, tvals + s, cnt, hist, run, wtmp);
        sl_long_pass<KV, BITS2, BITS1>(tkeys + s, tvals + s, keys + s, vals + s, cnt, hist, run, wtmp);
    }
}

// A whole sort by one workgroup: the passes of the long form, with the keys
// and values in registers and LDS between them.  A short sort is bound by
// latency.  Pairs, us, so and with two launches per pass: 1000 7.5 and 35, 4000
// 13 and 40, 8192 21 and 40, 12,000 28 and 42; with one pass of 8 bits, 8192
// 6.8 and 9.6.  At 16,384 the one CU is as slow (41 and 43).  Up to 8192 keys
// eight per lane: the longer kernel takes 3 us more at any length.
constexpr int kOneBlock = 1024, kOneRows = 8, kOneCap = 12 * kOneBlock;
struct OneSort {
    int n, begin, end, per;  // per: bits of a pass, at most 8
    uint32_t sign;           // flips the key's top bit
};
template <bool KV, int ROWS>
__global__ __launch_bounds__(kOneBlock) void k_sort_one(const uint32_t* kin, uint32_t* kout, const int32_t* vin,
                                                        int32_t* vout, OneSort g) {
    constexpr int W = kOneBlock / kWave;
    __shared__ uint32_t keys[ROWS * kOneBlock];
    __shared__ int32_t vals[KV ? ROWS * kOneBlock : 1];
    __shared__ alignas(16) uint16_t hist[W << 8];
    __shared__ uint32_t wtmp[W];
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int all = (g.n + kWave - 1) / kWave, per = all / W, rem = all % W;
    const int rows = per + (w < rem ? 1 : 0);
    const int e0 = (w * per + std::min(w, rem)) * kWave + lane_id();
    uint32_t x[ROWS], d[ROWS], old[ROWS], below[ROWS];
    int32_t v[ROWS];
    #pragma unroll
    for (int j = 0; j < ROWS; ++j) {
        const int e = e0 + j * kWave;
        const bool ok = j < rows && e < g.n;
        x[j] = ok ? kin[e] : 0u;
        if constexpr (KV) v[j] = ok ? vin[e] : 0;
    }
    for (int lo = g.begin; lo < g.end; lo += g.per) {
        const int bits = std::min(g.per, g.end - lo);
        // the last row's lanes past the end take the last digit: they stay the last ones
        #pragma unroll
        for (int j = 0; j < ROWS; ++j)
            d[j] = e0 + j * kWave < g.n ? __builtin_amdgcn_ubfe(x[j] ^ g.sign, lo, bits) : 255u;
        uint16_t* row = hist + (w << 8);
        sl_rank<8, 0, ROWS>(d, rows, row, old, below);
        sl_scan<8, kOneBlock>(hist, wtmp);
        #pragma unroll
        for (int j = 0; j < ROWS; ++j)
            if (j < rows) {
                const uint32_t p = row[d[j]] + old[j] + below[j];
                keys[p] = x[j];
                if constexpr (KV) vals[p] = v[j];
            }
        __syncthreads();
        #pragma unroll
        for (int j = 0; j < ROWS; ++j)
            if (j < rows) {
                x[j] = keys[e0 + j * kWave];
                if constexpr (KV) v[j] = vals[e0 + j * kWave];
            }
    }
    #pragma unroll
    for (int j = 0; j < ROWS; ++j) {
        const int e = e0 + j * kWave;
        if (j < rows && e < g.n) {
            kout[e] = x[j];
            if constexpr (KV) vout[e] = v[j];
        }
    }
}

template <bool KV, int BITS1, int BITS2>
void launch_sort_local(edpp_ctx* c, uint32_t* keys, int32_t* vals, uint32_t* tkeys, int32_t* tvals, const SlGeom& g) {
    const dim3 block(kSlBlock);
    hipLaunchKernelGGL((k_sort_local<KV, BITS1, BITS2>), dim3((unsigned)g.segs), block, 0, c->stream, keys, vals, g);
    hipLaunchKernelGGL((k_sort_long<KV, BITS1, BITS2>), dim3(4096), block, 0, c->stream, keys, vals, g);
    hipLaunchKernelGGL((k_sort_longer<KV, BITS1, BITS2>), dim3(512), block, 0, c->stream, keys, vals, tkeys, tvals, g);
}
template <bool KV>
void launch_sort_local(edpp_ctx* c, uint32_t* keys, int32_t* vals, uint32_t* tkeys, int32_t* tvals, const SlGeom& g) {
    if (g.segs == 1 << 16) launch_sort_local<KV, 8, 8>(c, keys, vals, tkeys, tvals, g);
    else if (g.segs == 1 << 15) launch_sort_local<KV, 9, 8>(c, keys, vals, tkeys, tvals, g);
    else launch_sort_local<KV, 9, 9>(c, keys, vals, tkeys, tvals, g);
}

// Before the passes: whether the keys' segments are short
int launch_sort_sample(edpp_ctx* c, const uint32_t* keys, const SlGeom& g) {
    hipLaunchKernelGGL(k_sort_sample, dim3(kSlSamples / 1024), dim3(1024), 0, c->stream, keys, g);
    EDPP_HIP(c, hipFuncSetAttribute((const void*)k_sort_decide, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * g.segs));
    hipLaunchKernelGGL(k_sort_decide, dim3(1), dim3(1024), (size_t)(2 * g.segs), c->stream, g);
    EDPP_HIP(c, hipGetLastError());
    return EDPP_OK;
}
// After them: keys (and vals, if any) in order of the top 16 bits; tkeys and tvals are spare
int launch_sort_local(edpp_ctx* c, uint32_t* keys, int32_t* vals, uint32_t* tkeys, int32_t* tvals, const SlGeom& g) {
    hipLaunchKernelGGL(k_sort_starts, dim3((unsigned)g.segs / 256 + 1), dim3(256), 0, c->stream, keys, g);
    if (vals) launch_sort_local<true>(c, keys, vals, tkeys, tvals, g);
    else launch_sort_local<false>(c, keys, vals, tkeys, tvals, g);
    EDPP_HIP(c, hipGetLastError());
    return EDPP_OK;
}

}  // namespace
}  // namespace edpp
