// gs_staged.hip — gather and scatter through windows of the random side, for
// tables that no XCD's L2 holds.
//
// Semantics are those of the pass loop of gather.hip (reference:
// opencl/primitives/gatherImpl.cpp:7-55, scatterImpl.cpp:9-54) for any pass
// count: out[i] = in[idx[i]] / out[idx[i]] = in[i] for idx[i] in [0, n), other
// indices skipped.
//
// A random 4-byte read of a table larger than an XCD's 4 MiB L2 fetches a
// 128-byte line (56 G lines/s at most, whatever holds them), and a random
// write leaves as a piece of a line.  Here the indices are first put in order
// of the window of the random side they fall in.  A gather then reads window
// after window, each from the L2 of the XCD that works on it, and brings the
// values back into index order; a scatter moves its values along, down to
// bins of 64 KiB of output, which it assembles in LDS.
//   gather:      k_st_probe     whether the indices are scattered at all
//   k_st_first   one read of the indices: chunks that are local, and a
//                gather's if they are not scattered, are done at once; the
//                others' elements are counted per window
//   k_st_groups, k_st_totals   prefixes of the counts
//   k_st_split   indices (scatter: and values) to window order, tile by tile
//                through LDS; a gather keeps each element's slot in its tile
//   gather:      k_st_gather    values, window after window
//                k_st_return    values back to their tiles and into order
//   scatter:     k_st_hist2, k_st_rows2, k_st_split2   a second split, of
//                               windows into bins
//                k_st_bins      every bin of the output through LDS
// The order of a window's elements is free, so ranks come from LDS counters
// (one atomic with return per element) and need no matching of lanes.
// (Random writes do not gather in an L2 as reads do: writing 2 MiB windows
// straight from window order sent 211 M write requests to memory for 2^28
// elements, where whole lines are 17 M, and took 2.9 ms against 1.7 ms for the
// second split and the bins.)
//
// 2^28 4-byte elements, random permutation, us per kernel: gather 186 (first)
// + 31 (prefixes) + 522 (split) + 1430 (gather: 290 M L2 requests, 204 G/s) +
// 587 (return); the others move 10 to 12 B per element at 4.6 to 5 TB/s;
// scatter 168 + 31 + 874 (split) + 254 (hist2) + 14 (rows2) + 880 (split2) +
// 580 (bins).
#include <algorithm>
#include "ctx.hpp"
#include "device.hpp"
#include "split_tile.hpp"
#include "window_tile.hpp"

namespace edpp {

namespace {

constexpr int64_t kStWindow = 2 << 20;    // bytes of the random side per window (an XCD's L2 holds 4 MiB)
constexpr int kStBin = 64 << 10;          // bytes of the output a scatter's workgroup assembles in LDS
constexpr int kStLocal = 4096;            // elements of a local chunk's LDS window

// Elements per 16-byte vector of T: 4 or 2.  A lane's step is one such vector
// of values (and 16 or 8 bytes of indices), so that a wave's accesses are
// contiguous for both widths.
template <class T>
constexpr int kStE = 16 / (int)sizeof(T);

// What every kernel of one call shares.  The indices are cut into chunks of
// 4096 and tiles of 64 KiB of values (4 or 2 chunks, kStEpl elements for each
// lane of the splits); lane t's elements [16h, 16h + 16) of a tile are vectors
// u*256 + t%256 of chunk 2h + t/256.
template <class T>
constexpr int kStEpl = 128 / (int)sizeof(T);
template <class T>
constexpr int kStTile = kStBlock * kStEpl<T>;
template <class T>
constexpr int kStCh = kStTile<T> / kStChunk;
// the lane's vector u of a tile: of its half h = u / (16/E)
template <class T>
__device__ __forceinline__ int64_t st_vec(int64_t tile, int u, uint32_t tid) {
    constexpr int E = kStE<T>;
    return tile * (kStTile<T> / E) + (int64_t)((u / (16 / E)) * (kStBlock / 256) + (int)(tid >> 8)) * (kStChunk / E) +
           u % (16 / E) * 256 + (tid & 255);
}
// whether the chunk of the lane's half h is finished, from st_done's bits
__device__ __forceinline__ bool st_skip(uint32_t mask, int h, uint32_t tid) {
    return (mask >> (h * (kStBlock / 256) + (int)(tid >> 8))) & 1u;
}
// lg bits of a line's number
__device__ __forceinline__ uint32_t st_line_hash(uint32_t line, int lg) { return (line * 0x9E3779B1u) >> (32 - lg); }
// finished chunks of a tile as bits (the last tile's missing ones among them)
template <int CH>
__device__ __forceinline__ uint32_t st_done(const StGeom& g, int64_t tile) {
    uint32_t m = 0;
    #pragma unroll
    for (int q = 0; q < CH; ++q) m |= (tile * CH + q >= g.chunks || g.done[tile * CH + q] ? 1u : 0u) << q;
    return m;
}

// Whether a gather's indices are scattered enough for the window order to pay.
// It takes 2750 us for 2^28 4-byte elements almost whatever the indices are,
// and a direct gather about 550 + 4900 d us, where d is the share of the
// elements that fetch a line of their own: two interleaved halves take 520 us,
// rows of 32 elements 530, 1000 distinct indices 910, a transposed 16384 x
// 16384 table 1700, random indices within 4 MiB 1800 (3360, 2080, 1720, 2080
// and 3410 in window order).  So d is measured: a workgroup takes
// kStProbeRows chunks that follow each other on one XCD (every kStProbeStep-th
// is on it), so that lines which its L2 keeps from one chunk to the next count
// once, as in the transposition, and counts their distinct lines in a bitmap
// of hashed line numbers, a quarter of the lines: 8192 elements in 2^16 bits,
// of which random ones set 0.94 each.  8 us.
constexpr int kStProbes = kWave;  // workgroups, spread evenly over the indices
constexpr int kStProbeRows = 8, kStProbeStep = 16, kStProbeLg = 16;
constexpr int kStProbeBlock = kStChunk / 4;
__global__ __launch_bounds__(kStProbeBlock) void k_st_probe(const int32_t* __restrict__ idx, StGeom g, int lg_line) {
    __shared__ uint32_t seen[1 << (kStProbeLg - 5)];
    __shared__ uint32_t wd[kStProbeBlock / kWave], wm[kStProbeBlock / kWave];
    const int t = threadIdx.x;
    const uint32_t nall = (uint32_t)g.n;
    constexpr int kSpan = (kStProbeRows - 1) * kStProbeStep + 1;
    const int64_t first = std::max<int64_t>(g.chunks - kSpan, 0) * blockIdx.x / (kStProbes - 1);
    uint32_t pos[kStProbeRows * 4];
    #pragma unroll
    for (int r = 0; r < kStProbeRows; ++r)
        st_load<uint32_t, 4>(reinterpret_cast<const uint32_t*>(idx), (first + r * kStProbeStep) * (kStChunk / 4) + t, g.n,
                             kStNone, pos + 4 * r);
    for (int i = t; i < (1 << (kStProbeLg - 5)); i += kStProbeBlock) seen[i] = 0;
    __syncthreads();
    uint32_t m = 0, d = 0;
    #pragma unroll
    for (int e = 0; e < kStProbeRows * 4; ++e)
        if (pos[e] < nall) {
            ++m;
            const uint32_t h = st_line_hash(pos[e] >> lg_line, kStProbeLg + 2);
            if ((h & 3u) == 0) atomicOr(seen + (h >> 7), 1u << ((h >> 2) & 31));
        }
    __syncthreads();
    for (int i = t; i < (1 << (kStProbeLg - 5)); i += kStProbeBlock) d += __popc(seen[i]);
    d = wave_sum(d);
    m = wave_sum(m);
    if (lane_id() == 0) {
        wd[t / kWave] = d;
        wm[t / kWave] = m;
    }
    __syncthreads();
    if (t < kWave) {
        d = wave_sum(t < kStProbeBlock / kWave ? wd[t] : 0u);
        m = wave_sum(t < kStProbeBlock / kWave ? wm[t] : 0u);
        if (t == 0) {
            g.probe[2 * blockIdx.x] = 4 * d;
            g.probe[2 * blockIdx.x + 1] = m;
        }
    }
}
// The line lies where the window order is the faster one for certain: random
// indices within 16 MiB (d = 0.87, direct 3700, in window order 2790 us) and
// Zipf(0.8) ones (4710, 2730) are above it; below it, random ones within 8 MiB
// (0.76: 2700, 3000), and Zipf(1) ones (0.6: 2930 and 2600, but 8-byte values
// 1490 and 1770).  The same in every wave.
__device__ __forceinline__ bool st_scattered(const StGeom& g) {
    const uint2 y = reinterpret_cast<const uint2*>(g.probe)[lane_id()];
    return wave_sum(y.x) * 16u > wave_sum(y.y) * 13u;
}

// One chunk per workgroup, of as many lanes as give a CU 32 waves beside the
// LDS windows.  A chunk whose indices fall inside kStLocal elements (a
// block-local permutation) goes through an LDS window: a gather loads the
// window with consecutive loads and reads its values from LDS; a scatter
// writes its values into the window and stores the covered positions as runs.
// A gather addresses a chunk directly if its indices fall inside g.near
// elements, as L2 holds that many, and every chunk if the indices are not
// scattered.  A scatter does so with a chunk that writes at least kStCover
// sixteenths of the lines it touches, and soon (its first quarter, of 8-byte
// values half, touches at most 3 lines per 16 elements), or whole 32-byte
// sectors by neighbouring lanes, as most of that leaves L2 as whole lines or
// sectors.  The others are counted.
//
// Scatters of 2^28 4-byte elements, us in one direct pass / in four / in
// window order: two interleaved streams 590 / 1610 / 2690, 64 of them 1150 /
// 1880 / 2680, rows of 32 elements 670 / 1910 / 2610, every second element
// 1310 / 2160 / 2700, rows of 8 1950 / 2610 / 2740; but every eighth element
// 6710 / 5480 / 2690, rows of 2 5620 / 3560 / 2770, 256 interleaved streams
// 3940 / 3800 / 3090, of random lengths 3210 / 2530 / 2730.  Lines are counted
// by hash in bytes of LDS; where the indices are scattered, the first part's
// are too many already (k_st_first of a random scatter 168 us, 183 with all
// lines counted, 162 without).  A scatter's lanes
// take 4 elements per step also of 8-byte values, so that the lanes of one
// store touch fewer streams (128 streams 1240 us, by steps of 2 2040); a
// gather's stores have to be consecutive (470, by steps of 4 820).
constexpr uint32_t kStCover = 7;
constexpr int kStLineLg = 12;
template <class T>
constexpr int kStFirstBlock = 64 * (int)sizeof(T);  // 256 or 512
template <class T, bool SC>
__global__ __launch_bounds__(kStFirstBlock<T>) void k_st_first(const T* __restrict__ in, T* __restrict__ out,
                                                  const int32_t* __restrict__ idx, StGeom g) {
    constexpr int E = kStE<T>;
    constexpr int BL = kStFirstBlock<T>;
    constexpr int NW = BL / kWave;
    constexpr int N = kStChunk / BL;  // elements per lane, in steps of P
    constexpr int P = SC ? 4 : E;
    extern __shared__ uint32_t cnt[];  // [W << cl]
    __shared__ __attribute__((aligned(16))) T win[kStLocal];
    uint8_t* seen = reinterpret_cast<uint8_t*>(win);  // [1 << kStLineLg] of a scatter that fills no window
    __shared__ uint32_t wlo[NW], whi[NW], wsw[SC ? NW : 1];
    __shared__ uint32_t cov[SC ? kStLocal / 32 : 1];
    const int t = threadIdx.x, w = t / kWave;
    const int64_t v0 = (int64_t)blockIdx.x * (kStChunk / P) + t;
    const uint32_t nall = (uint32_t)g.n;
    uint32_t pos[N];
    T val[N];
    #pragma unroll
    for (int u = 0; u < N / P; ++u)
        st_load<uint32_t, P>(reinterpret_cast<const uint32_t*>(idx), v0 + u * BL, g.n, kStNone, pos + P * u);
    const bool scattered = SC || st_scattered(g);
    const int cl = st_copies_lg(g.W);
    for (int i = t; i < (g.WP << cl); i += BL) cnt[i] = 0;
    if (SC) {
        for (int i = t; i < kStLocal / 32; i += BL) cov[i] = 0;
        for (int i = t; i < (1 << kStLineLg) / 4; i += BL) reinterpret_cast<uint32_t*>(win)[i] = 0;
    }
    uint32_t lo = kStNone, hi = 0;
    #pragma unroll
    for (int e = 0; e < N; ++e)
        if (pos[e] < nall) {
            lo = std::min(lo, pos[e]);
            hi = std::max(hi, pos[e]);
        }
    lo = ~wave_max(~lo);
    hi = wave_max(hi);
    constexpr int kLgLine = sizeof(T) == 4 ? 5 : 4;
    uint32_t broken = 0;  // the wave's lane steps (4-byte elements: pairs of lanes) that touch more than one sector
    if constexpr (SC) {
        #pragma unroll
        for (int u = 0; u < N / P; ++u) {
            uint32_t x = 0;
            #pragma unroll
            for (int k = 1; k < P; ++k) x |= pos[P * u] ^ pos[P * u + k];
            if (sizeof(T) == 4) x |= pos[P * u] ^ (uint32_t)__builtin_amdgcn_mov_dpp((int)pos[P * u], 0xB1, 0xf, 0xf, true);
            broken += __popcll(ballot(x >> (kLgLine - 2) != 0));
        }
    }
    if (lane_id() == 0) {
        wlo[w] = lo;
        whi[w] = hi;
        if (SC) wsw[w] = broken;
    }
    __syncthreads();
    #pragma unroll
    for (int x = 0; x < NW; ++x) {
        lo = std::min(lo, wlo[x]);
        hi = std::max(hi, whi[x]);
    }
    // the same in the whole workgroup from here on
    const bool some = lo <= hi;
    const bool window = some && hi - lo < (uint32_t)kStLocal;
    bool near = !some || window;
    if constexpr (SC) {
        broken = 0;
        #pragma unroll
        for (int x = 0; x < NW; ++x) broken += wsw[x];
        near = near || 8 * broken <= kStChunk / P;
        // distinct lines, by hash (a few hundred where it matters), first of the
        // chunk's leading elements
        auto lines = [&](int e0, int e1) {
            #pragma unroll
            for (int e = 0; e < N; ++e)
                if (e >= e0 && e < e1 && pos[e] < nall) seen[st_line_hash(pos[e] >> kLgLine, kStLineLg)] = 1;
            __syncthreads();
            uint32_t d = 0;
            #pragma unroll
            for (int i = 0; i < (1 << kStLineLg) / 16 / kWave; ++i) {
                const v4u32 y = reinterpret_cast<const v4u32*>(seen)[i * kWave + lane_id()];
                d += __popc(y[0]) + __popc(y[1]) + __popc(y[2]) + __popc(y[3]);
            }
            return wave_sum(d);  // every wave sums all of them
        };
        const uint32_t m = (uint32_t)std::min<int64_t>(g.n - (int64_t)blockIdx.x * kStChunk, kStChunk);
        if (!near && lines(0, P) * 16u <= 3u * (BL * P)) {
            __syncthreads();
            near = (lines(P, N) << kLgLine) * kStCover <= 16u * m;
        }
    } else {
        near = near || hi - lo < g.near || !scattered;
    }
    if (t == 0) {
        g.done[blockIdx.x] = near ? 1 : 0;
        // read first, and many words: one address that every workgroup stores
        // to takes them one after the other (35 us at 2^23 elements)
        uint32_t* w = st_gate(g, blockIdx.x);
        if (!near && ld_relaxed(w) == 0) st_relaxed(w, 1u);
    }
    if (!near) {
        const uint32_t copy = t & ((1u << cl) - 1u);
        #pragma unroll
        for (int e = 0; e < N; ++e)
            if (pos[e] < nall)
                __hip_atomic_fetch_add(cnt + ((pos[e] >> g.shift) << cl) + copy, 1u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
        uint32_t* row = reinterpret_cast<uint32_t*>(g.count + (int64_t)blockIdx.x * g.WP);
        for (int i = t; i < g.WP / 2; i += BL) {
            uint32_t a = 0, b = 0;
            for (int c = 0; c < (1 << cl); ++c) {
                a += cnt[((2 * i) << cl) + c];
                b += cnt[((2 * i + 1) << cl) + c];
            }
            row[i] = a | (b << 16);
        }
        return;
    }
    if constexpr (SC) {
        #pragma unroll
        for (int u = 0; u < N / E; ++u)
            st_load<T, E>(in, (v0 + u / (P / E) * BL) * (P / E) + u % (P / E), g.n, T(0), val + E * u);
        if (window) {
            #pragma unroll
            for (int e = 0; e < N; ++e)
                if (pos[e] < nall) {
                    const uint32_t o = pos[e] - lo;
                    win[o] = val[e];
                    atomicOr(cov + (o >> 5), 1u << (o & 31));
                }
            __syncthreads();
            for (uint32_t o = t; o <= hi - lo; o += BL)
                if ((cov[o >> 5] >> (o & 31)) & 1u) out[lo + o] = win[o];
        } else {
            #pragma unroll
            for (int e = 0; e < N; ++e)
                if (pos[e] < nall) out[pos[e]] = val[e];
        }
    } else {
        if (window) {
            for (uint32_t o = t; o <= hi - lo; o += BL) win[o] = in[lo + o];
            __syncthreads();
            #pragma unroll
            for (int e = 0; e < N; ++e) val[e] = pos[e] < nall ? win[pos[e] - lo] : T(0);
        } else {
            #pragma unroll
            for (int e = 0; e < N; ++e) val[e] = pos[e] < nall ? in[pos[e]] : T(0);
        }
        #pragma unroll
        for (int u = 0; u < N / E; ++u) {
            bool ok[E];
            #pragma unroll
            for (int k = 0; k < E; ++k) ok[k] = pos[E * u + k] < nall;
            st_store<T, E>(out, v0 + u * BL, val + E * u, ok);
        }
    }
}

// LDS of the two splits: [S] indices, then [S] values through the same
// buffer; counts and offsets of the buckets
template <class T, bool SC>
constexpr size_t st_split_lds() {
    return (size_t)kStTile<T> * (SC ? sizeof(T) : 4) + 8 * kStBuckets;
}

// Bucket of an element among B from b0 on; B for one that is none (its shift
// is above every window: n < 2^31)
__device__ __forceinline__ uint32_t st_bucket(uint32_t x, int shift, uint32_t b0, uint32_t B) {
    return std::min((x >> shift) - b0, B);
}

// The m slots' indices to their output positions d[] (slot + dlt[bucket]; past
// the output, where the store is dropped, for the slots of no element)
template <int EPL>
__device__ __forceinline__ void st_put_index(uint32_t tid, uint32_t m, const uint32_t* buf, const uint32_t* dlt,
                                             int shift, uint32_t b0, int B, const BufSink<uint32_t>& out,
                                             uint32_t (&d)[EPL]) {
    #pragma unroll
    for (int j = 0; j < EPL; ++j) {
        const uint32_t i = tid + j * kStBlock;
        const uint32_t k = buf[i];
        const uint32_t p = dlt[st_bucket(k, shift, b0, (uint32_t)B)] + i;
        d[j] = i < m ? p : kStNone;
        out.put(d[j], k);
    }
}

// The lane's elements of a tile of p (T: the values' type, which sets the
// layout); in the last tile through a buffer descriptor that ends at n (loads
// past it read 0)
template <class T, class V>
__device__ __forceinline__ void st_load_tile(const V* __restrict__ p, int64_t tile, int64_t n, uint32_t tid,
                                             V (&x)[kStEpl<T>]) {
    constexpr int E = kStE<T>;
    if ((tile + 1) * kStTile<T> <= n) {
        typedef V vec __attribute__((ext_vector_type(E)));
        #pragma unroll
        for (int u = 0; u < kStEpl<T> / E; ++u) {
            const vec v = ld_stream(reinterpret_cast<const vec*>(p) + st_vec<T>(tile, u, tid));
            #pragma unroll
            for (int k = 0; k < E; ++k) x[E * u + k] = v[k];
        }
    } else {
        const int64_t e0 = tile * kStTile<T>;
        const __amdgpu_buffer_rsrc_t r = buf_rsrc(p + e0, n - e0);
        const uint32_t l = (tid >> 8) * kStChunk + (tid & 255) * E;
        #pragma unroll
        for (int e = 0; e < kStEpl<T>; ++e)
            x[e] = buf_load<V>(r, l * (uint32_t)sizeof(V),
                               (uint32_t)((e / 16 * (kStBlock / 256) * kStChunk + e % 16 / E * 256 * E + e % E) * sizeof(V)));
    }
}
// its indices, kStNone for none
template <class T>
__device__ __forceinline__ void st_load_idx(const int32_t* __restrict__ idx, int64_t tile, int64_t n, uint32_t mask,
                                            uint32_t tid, uint32_t (&x)[kStEpl<T>]) {
    constexpr int E = kStE<T>;
    const uint32_t nall = (uint32_t)n;
    st_load_tile<T, uint32_t>(reinterpret_cast<const uint32_t*>(idx), tile, n, tid, x);
    // elements of the tile before n, less the lane's first one
    const int left = (int)std::min<int64_t>(n - tile * kStTile<T>, kStTile<T>) -
                     (int)((tid >> 8) * kStChunk + (tid & 255) * E);
    #pragma unroll
    for (int e = 0; e < kStEpl<T>; ++e) {
        const int l = st_skip(mask, e / 16, tid) ? 0 : left;
        x[e] = e / 16 * (kStBlock / 256) * kStChunk + e % 16 / E * 256 * E + e % E < l && x[e] < nall ? x[e] : kStNone;
    }
}

// Indices (and a scatter's values) of one tile to window order: sidx / sval
// [base[w] + gsum[w] + rows[w] ...].  A gather's element keeps its slot in the
// window-ordered tile in slot[].
template <class T, bool SC>
__global__ __launch_bounds__(kStBlock, kStBlock / 128) void k_st_split(const T* __restrict__ in,
                                                                       const int32_t* __restrict__ idx, StGeom g,
                                                                       uint32_t* __restrict__ sidx, T* __restrict__ sval,
                                                                       uint16_t* __restrict__ slot) {
    constexpr int CH = kStCh<T>;
    constexpr int E = kStE<T>;
    constexpr int EPL = kStEpl<T>;
    extern __shared__ char smem[];
    uint32_t* buf = reinterpret_cast<uint32_t*>(smem);
    T* vbuf = reinterpret_cast<T*>(smem);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(smem + (size_t)kStTile<T> * (SC ? sizeof(T) : 4));
    uint32_t* off = cnt + kStBuckets;
    __shared__ uint32_t wtmp[kStBlock / kWave];
    if (*g.open == 0) return;
    const uint32_t tid = threadIdx.x;
    if (blockIdx.x == 0) st_keep_bases<CH>(g, tid, wtmp, off);
    const int64_t tile = st_order(blockIdx.x, (uint32_t)g.tiles, g.xcds);
    const uint32_t mask = st_done<CH>(g, tile);
    if (mask == (1u << CH) - 1u) return;
    const int cl = st_copies_lg(g.W);
    uint32_t at[EPL / 2], m;
    {
        uint32_t x[EPL];
        st_load_idx<T>(idx, tile, g.n, mask, tid, x);
        m = st_rank<EPL>(tid, x, at, [&](int, uint32_t v) { return st_bucket(v, g.shift, 0u, (uint32_t)g.W); }, g.W, cl, cnt, off, wtmp);
        st_place<uint32_t, EPL>(buf, at, x);
    }
    if (!SC) {
        // the workspace holds whole tiles
        #pragma unroll
        for (int u = 0; u < EPL / E; ++u) {
            if (st_skip(mask, u / (16 / E), tid)) continue;
            if constexpr (E == 4)
                st_stream((uint64_t)at[2 * u + 1] << 32 | at[2 * u], reinterpret_cast<uint64_t*>(slot) + st_vec<T>(tile, u, tid));
            else
                st_stream(at[u], reinterpret_cast<uint32_t*>(slot) + st_vec<T>(tile, u, tid));
        }
    }
    __syncthreads();
    st_distances(g, tile, tid, cl, cnt, off, wtmp);
    T val[EPL];
    if (SC) st_load_tile<T, T>(in, tile, g.n, tid, val);
    __syncthreads();
    uint32_t d[EPL];
    st_put_index<EPL>(tid, m, buf, cnt, g.shift, 0u, g.W, buf_sink(sidx, g.n), d);
    if constexpr (SC) {
        __syncthreads();
        st_place<T, EPL>(vbuf, at, val);
        __syncthreads();
        const BufSink<T> sink = buf_sink(sval, g.n);
        #pragma unroll
        for (int j = 0; j < EPL; ++j) sink.put(d[j], vbuf[tid + j * kStBlock]);
    }
}

// A second-level tile: elements [lo, hi) of one window's stretch of the
// window order; t is its number among the window's nt tiles.
struct StTile2 {
    int w;
    uint32_t lo, hi, t, nt;
};
template <int S>
__device__ __forceinline__ void st_tile2(const StGeom& g, uint32_t tile, StTile2& r) {
    const int a = g.win2[tile];
    r.w = a;
    r.t = tile - g.tile2[a];
    r.nt = g.tile2[a + 1] - g.tile2[a];
    r.lo = g.base[a] + r.t * (uint32_t)S;
    r.hi = std::min(r.lo + (uint32_t)S, g.base[a + 1]);
}

// bin counts of the second-level tiles
template <class T>
__global__ __launch_bounds__(kStBlock) void k_st_hist2(StGeom g, const uint32_t* __restrict__ sidx) {
    constexpr int S = kStTile<T>;
    __shared__ uint32_t cnt[kStBuckets];
    if (*g.open == 0) return;
    const uint32_t tiles = g.tile2[g.W];
    if (blockIdx.x >= tiles) return;
    const int B = 1 << g.lg_subs;
    const int cl = st_copies_lg(B);
    StTile2 r;
    st_tile2<S>(g, st_order(blockIdx.x, tiles, g.xcds), r);
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(sidx + r.lo, r.hi - r.lo);
    uint32_t x[kStEpl<T>];
    #pragma unroll
    for (int j = 0; j < kStEpl<T>; ++j) x[j] = buf_load<uint32_t>(rs, threadIdx.x * 4, j * kStBlock * 4);
    for (int i = threadIdx.x; i < (B << cl); i += kStBlock) cnt[i] = 0;
    __syncthreads();
    const uint32_t b0 = (uint32_t)r.w << g.lg_subs, copy = threadIdx.x & ((1u << cl) - 1u);
    #pragma unroll
    for (int j = 0; j < kStEpl<T>; ++j)
        if (threadIdx.x + j * kStBlock < r.hi - r.lo)
            __hip_atomic_fetch_add(cnt + (((x[j] >> g.sub_shift) - b0) << cl) + copy, 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    uint32_t* rows = g.rows2 + ((int64_t)g.tile2[r.w] << g.lg_subs) + r.t;
    for (int i = threadIdx.x; i < B; i += kStBlock) {
        uint32_t s = 0;
        for (int c = 0; c < (1 << cl); ++c) s += cnt[(i << cl) + c];
        rows[(int64_t)i * r.nt] = s;
    }
}

// exclusive prefix over the workgroup's lanes of s, plus carry; carry grows by
// the sum.  wt: one word per wave.  Two barriers.
template <int BLOCK>
__device__ __forceinline__ uint32_t st_block_prefix(uint32_t s, uint32_t* wt, uint32_t& carry) {
    const int w = threadIdx.x / kWave;
    const uint32_t inc = wave_inclusive_add(s);
    if (lane_id() == kWave - 1) wt[w] = inc;
    __syncthreads();
    uint32_t before = carry, all = 0;
    #pragma unroll
    for (int q = 0; q < BLOCK / kWave; ++q) {
        before += q < w ? wt[q] : 0u;
        all += wt[q];
    }
    carry += all;
    __syncthreads();
    return before + inc - s;
}

// One window's bin counts become output positions; the bins' first positions
__global__ __launch_bounds__(kStRowBlock) void k_st_rows2(StGeom g) {
    __shared__ uint32_t wt[kStRowBlock / kWave];
    if (*g.open == 0) return;
    const int w = blockIdx.x;
    const uint32_t nt = g.tile2[w + 1] - g.tile2[w];
    uint32_t* rows = g.rows2 + ((int64_t)g.tile2[w] << g.lg_subs);
    const int64_t len = (int64_t)nt << g.lg_subs;
    uint32_t carry = g.base[w];
    if (nt == 0)
        for (int i = threadIdx.x; i < (1 << g.lg_subs); i += kStRowBlock) g.bins[((int64_t)w << g.lg_subs) + i] = carry;
    for (int64_t b = 0; b < len; b += kStRowBlock * 4) {
        uint32_t x[4], s = 0;
        const int64_t i0 = b + (int64_t)threadIdx.x * 4;
        #pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = i0 + k < len ? rows[i0 + k] : 0u;
            s += x[k];
        }
        uint32_t y = st_block_prefix<kStRowBlock>(s, wt, carry);
        #pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (i0 + k < len) {
                rows[i0 + k] = y;
                if ((i0 + k) % nt == 0) g.bins[((int64_t)w << g.lg_subs) + (i0 + k) / nt] = y;
            }
            y += x[k];
        }
    }
}

// One second-level tile to bin order
template <class T>
__global__ __launch_bounds__(kStBlock, kStBlock / 128) void k_st_split2(StGeom g, const uint32_t* __restrict__ sidx,
                                                                        const T* __restrict__ sval,
                                                                        uint32_t* __restrict__ didx,
                                                                        T* __restrict__ dval) {
    constexpr int S = kStTile<T>;
    constexpr int EPL = kStEpl<T>;
    extern __shared__ char smem[];
    uint32_t* buf = reinterpret_cast<uint32_t*>(smem);
    T* vbuf = reinterpret_cast<T*>(smem);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(smem + (size_t)S * sizeof(T));
    uint32_t* off = cnt + kStBuckets;
    __shared__ uint32_t wtmp[kStBlock / kWave];
    if (*g.open == 0) return;
    const uint32_t tiles = g.tile2[g.W];
    if (blockIdx.x >= tiles) return;
    const int B = 1 << g.lg_subs;
    const int cl = st_copies_lg(B);
    StTile2 r;
    st_tile2<S>(g, st_order(blockIdx.x, tiles, g.xcds), r);
    const uint32_t b0 = (uint32_t)r.w << g.lg_subs;
    const uint32_t have = r.hi - r.lo;
    const uint32_t tid = threadIdx.x;
    uint32_t at[EPL / 2];
    {
        uint32_t x[EPL];
        const __amdgpu_buffer_rsrc_t rs = buf_rsrc(sidx + r.lo, have);
        #pragma unroll
        for (int j = 0; j < EPL; ++j) x[j] = buf_load<uint32_t>(rs, tid * 4, j * kStBlock * 4);
        #pragma unroll
        for (int j = 0; j < EPL; ++j) x[j] = tid + j * kStBlock < have ? x[j] : kStNone;
        st_rank<EPL>(tid, x, at, [&](int, uint32_t v) { return st_bucket(v, g.sub_shift, b0, (uint32_t)B); }, B, cl, cnt, off, wtmp);
        st_place<uint32_t, EPL>(buf, at, x);
    }
    __syncthreads();
    const uint32_t* rows = g.rows2 + ((int64_t)g.tile2[r.w] << g.lg_subs) + r.t;
    for (int i = (int)tid; i < B; i += kStBlock) cnt[i] = rows[(int64_t)i * r.nt] - off[i << cl];
    T val[EPL];
    const __amdgpu_buffer_rsrc_t rv = buf_rsrc(sval + r.lo, have);
    #pragma unroll
    for (int j = 0; j < EPL; ++j) val[j] = buf_load<T>(rv, tid * (uint32_t)sizeof(T), j * kStBlock * (uint32_t)sizeof(T));
    __syncthreads();
    uint32_t d[EPL];
    st_put_index<EPL>(tid, have, buf, cnt, g.sub_shift, b0, B, buf_sink(didx, g.n), d);
    __syncthreads();
    st_place<T, EPL>(vbuf, at, val);
    __syncthreads();
    const BufSink<T> sink = buf_sink(dval, g.n);
    #pragma unroll
    for (int j = 0; j < EPL; ++j) sink.put(d[j], vbuf[tid + j * kStBlock]);
}

// out[didx[j]] = dval[j] for one bin of kStBin bytes of the output, through
// LDS: every covered line leaves whole
constexpr int kStBinBlock = 1024;
template <class T>
__global__ __launch_bounds__(kStBinBlock, kStBinBlock / 128) void k_st_bins(StGeom g, int64_t nbins,
                                                                            const uint32_t* __restrict__ didx,
                                                                            const T* __restrict__ dval,
                                                                            T* __restrict__ out) {
    constexpr int E = kStBin / (int)sizeof(T);
    extern __shared__ char smem[];
    T* win = reinterpret_cast<T*>(smem);                              // [E]
    uint32_t* cov = reinterpret_cast<uint32_t*>(smem + kStBin);       // [E / 32]
    if (*g.open == 0) return;
    st_close(g);
    for (uint32_t ob = blockIdx.x; ob < (uint32_t)nbins; ob += gridDim.x) {
    const int64_t bin = st_order(ob, (uint32_t)nbins, g.xcds);
    const uint32_t m = std::min<uint32_t>(g.base[g.W], (uint32_t)g.n);
    const uint32_t lo = std::min(g.bins[bin], m), hi = bin + 1 < nbins ? std::min(g.bins[bin + 1], m) : m;
    if (lo >= hi) continue;  // the same in the whole workgroup
    const uint32_t o0 = (uint32_t)bin * (uint32_t)E;
    for (int i = threadIdx.x; i < E / 32; i += kStBinBlock) cov[i] = 0;
    __syncthreads();
    for (uint32_t b = lo; b < hi; b += kStBinBlock * 8) {
        uint32_t x[8];
        T v[8];
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t e = b + threadIdx.x + j * kStBinBlock;
            x[j] = e < hi ? ld_stream(didx + e) : kStNone;
            v[j] = e < hi ? ld_stream(dval + e) : T(0);
        }
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t o = x[j] - o0;
            if (o < (uint32_t)E) {
                win[o] = v[j];
                atomicOr(cov + (o >> 5), 1u << (o & 31));
            }
        }
    }
    __syncthreads();
    constexpr int V = kStE<T>;
    for (int q = threadIdx.x; q < E / V; q += kStBinBlock) {
        const uint32_t c = cov[q / (32 / V)] >> (V * (q % (32 / V)));
        T v[V];
        bool ok[V];
        #pragma unroll
        for (int k = 0; k < V; ++k) {
            v[k] = win[V * q + k];
            ok[k] = (c >> k) & 1u;  // positions at or past n are never covered
        }
        st_store<T, V>(out, (int64_t)(o0 / V) + q, v, ok);
    }
    __syncthreads();
    }
}

// sval[j] = in[sidx[j]]: workgroups of one XCD walk one range of the window
// order, so the windows being read at one time are few and stay in its L2.
// 4-byte values take their indices' place: a lane has read all of its indices
// before it stores.
template <class T>
constexpr int kStGe = 128 / (int)sizeof(T);  // staged elements per lane
template <class T>
constexpr int kStPart = 256 * kStGe<T>;      // and per workgroup
template <class T>
__global__ __launch_bounds__(256) void k_st_gather(const T* __restrict__ in, StGeom g, const uint32_t* sidx, T* sval) {
    constexpr int E = kStE<T>;
    if (*g.open == 0) return;
    const int64_t m = std::min<int64_t>(g.base[g.W], g.n);
    const uint32_t parts = (uint32_t)((m + kStPart<T> - 1) / kStPart<T>);
    if (blockIdx.x >= parts) return;
    const int64_t v0 = (int64_t)st_order(blockIdx.x, parts, g.xcds) * (kStPart<T> / E) + threadIdx.x;
    const uint32_t nall = (uint32_t)g.n;
    uint32_t pos[kStGe<T>];
    T val[kStGe<T>];
    #pragma unroll
    for (int u = 0; u < kStGe<T> / E; ++u) st_load<uint32_t, E>(sidx, v0 + u * 256, m, kStNone, pos + E * u);
    #pragma unroll
    for (int e = 0; e < kStGe<T>; ++e) val[e] = pos[e] < nall ? in[pos[e]] : T(0);
    #pragma unroll
    for (int u = 0; u < kStGe<T> / E; ++u) {
        bool ok[E];
        #pragma unroll
        for (int k = 0; k < E; ++k) ok[k] = E * (v0 + u * 256) + k < m;
        st_store<T, E>(sval, v0 + u * 256, val + E * u, ok);
    }
}

// A gather's values back into order: the tile's runs of sval are copied to
// LDS slot by slot, then every element takes its slot's value.  first[] holds
// the window of every kStStep-th slot; runs are longer than that on average,
// so two steps from there reach a slot's window but for a few.
constexpr int kStStep = 8;
template <class T>
constexpr size_t st_return_lds() {
    return (size_t)kStTile<T> * sizeof(T) + 8 * kStBuckets + kStTile<T> / kStStep * 2;
}
template <class T>
__global__ __launch_bounds__(kStBlock, kStBlock / 128) void k_st_return(T* __restrict__ out, StGeom g,
                                                                        const T* __restrict__ sval,
                                                                        const uint16_t* __restrict__ slot) {
    constexpr int CH = kStCh<T>;
    constexpr int E = kStE<T>;
    constexpr int EPL = kStEpl<T>;
    extern __shared__ char smem[];
    T* vbuf = reinterpret_cast<T*>(smem);                                                // [tile]
    uint32_t* end = reinterpret_cast<uint32_t*>(smem + (size_t)kStTile<T> * sizeof(T));  // [W] counts, then slot ends
    uint32_t* dlt = end + kStBuckets;                                 // [W] slot starts, then slot to position
    uint16_t* first = reinterpret_cast<uint16_t*>(dlt + kStBuckets);  // [tile / kStStep]
    __shared__ uint32_t wtmp[kStBlock / kWave];
    if (*g.open == 0) return;
    st_close(g);
    const uint32_t nall = (uint32_t)g.n;
    const int64_t tile = st_order(blockIdx.x, (uint32_t)g.tiles, g.xcds);
    const uint32_t mask = st_done<CH>(g, tile);
    if (mask == (1u << CH) - 1u) return;
    const uint32_t tid = threadIdx.x;
    uint32_t sl[EPL / 2];  // two slots per word
    #pragma unroll
    for (int u = 0; u < EPL / E; ++u) {
        const bool skip = st_skip(mask, u / (16 / E), tid);
        if constexpr (E == 4) {
            const uint64_t p = skip ? ~0ull : ld_stream(reinterpret_cast<const uint64_t*>(slot) + st_vec<T>(tile, u, tid));
            sl[2 * u] = (uint32_t)p;
            sl[2 * u + 1] = (uint32_t)(p >> 32);
        } else {
            sl[u] = skip ? ~0u : ld_stream(reinterpret_cast<const uint32_t*>(slot) + st_vec<T>(tile, u, tid));
        }
    }
    for (int i = (int)tid; i < g.W; i += kStBlock) {
        uint32_t s = 0;
        #pragma unroll
        for (int q = 0; q < CH; ++q)  // chunks past the last one are marked done
            if (!((mask >> q) & 1u)) s += g.count[(tile * CH + q) * g.WP + i];
        end[i] = std::min<uint32_t>(s, (uint32_t)kStTile<T>);
    }
    const uint32_t m = std::min<uint32_t>(st_scan(tid, end, dlt, g.W, wtmp), (uint32_t)kStTile<T>);
    for (int i = (int)tid; i < g.W; i += kStBlock) {
        const uint32_t a = dlt[i], e = std::min<uint32_t>(a + end[i], (uint32_t)kStTile<T>);
        for (uint32_t k = (a + kStStep - 1) / kStStep; k * kStStep < e; ++k) first[k] = (uint16_t)i;
        end[i] = e;
        dlt[i] = g.base[i] + g.gsum[tile / g.group * g.WP + i] + g.rows[tile * g.WP + i] - a;
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(sval, g.n);
    #pragma unroll
    for (int h = 0; h < EPL; h += 8) {  // eight slots at a time
        uint32_t w[8];
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t i = tid + (h + j) * kStBlock;
            w[j] = first[std::min(i, m - 1) / kStStep];  // m > 0: some chunk is not finished
        }
        #pragma unroll
        for (int r = 0; r < 2; ++r)
            #pragma unroll
            for (int j = 0; j < 8; ++j)
                w[j] += std::min<uint32_t>(tid + (h + j) * kStBlock, m - 1) >= end[w[j]] ? 1u : 0u;
        T v[8];
        #pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t i = std::min<uint32_t>(tid + (h + j) * kStBlock, m - 1);
            while (i >= end[w[j]]) ++w[j];  // ends at the latest at the last window, whose end is m
            v[j] = buf_load<T>(rs, std::min(dlt[w[j]] + i, nall) * (uint32_t)sizeof(T));
        }
        #pragma unroll
        for (int j = 0; j < 8; ++j) vbuf[tid + (h + j) * kStBlock] = v[j];
    }
    __syncthreads();
    #pragma unroll
    for (int u = 0; u < EPL / E; ++u) {
        T y[E];
        bool ok[E];
        #pragma unroll
        for (int k = 0; k < E; ++k) {
            const int e = E * u + k;
            const uint32_t s = e & 1 ? sl[e / 2] >> 16 : sl[e / 2] & 0xFFFFu;
            ok[k] = s < m;
            y[k] = vbuf[ok[k] ? s : 0u];
        }
        st_store<T, E>(out, st_vec<T>(tile, u, tid), y, ok);
    }
}

struct StBufs {
    uint32_t *sidx, *didx;  // window order; a scatter's bin order
    void *sval, *dval;
    uint16_t* slot;
};

template <class T, bool SC>
int run_staged(edpp_ctx* c, const T* in, T* out, const int32_t* idx, const StGeom& g, const StBufs& b, int64_t nbins) {
    constexpr int CH = kStCh<T>;
    const unsigned grid = (unsigned)g.tiles;
    constexpr size_t l3 = st_split_lds<T, SC>();
    const size_t l1 = ((size_t)g.WP << st_copies_lg(g.W)) * 4;
    T* sval = static_cast<T*>(b.sval);
    if (!SC)
        hipLaunchKernelGGL(k_st_probe, dim3(kStProbes), dim3(kStProbeBlock), 0, c->stream, idx, g, sizeof(T) == 4 ? 5 : 4);
    EDPP_HIP(c, hipFuncSetAttribute((const void*)k_st_split<T, SC>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l3));
    hipLaunchKernelGGL((k_st_first<T, SC>), dim3((unsigned)g.chunks), dim3(kStFirstBlock<T>), l1, c->stream, in, out, idx, g);
    launch_st_prefix<CH>(c->stream, g, nullptr);
    hipLaunchKernelGGL((k_st_split<T, SC>), dim3(grid), dim3(kStBlock), l3, c->stream, in, idx, g, b.sidx, sval, b.slot);
    if constexpr (SC) {
        const unsigned grid2 = (unsigned)(g.tiles + g.W);  // a window's last tile may be short
        T* dval = static_cast<T*>(b.dval);
        EDPP_HIP(c, hipFuncSetAttribute((const void*)k_st_split2<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l3));
        hipLaunchKernelGGL((k_st_hist2<T>), dim3(grid2), dim3(kStBlock), 0, c->stream, g, (const uint32_t*)b.sidx);
        hipLaunchKernelGGL(k_st_rows2, dim3((unsigned)g.W), dim3(kStRowBlock), 0, c->stream, g);
        hipLaunchKernelGGL((k_st_split2<T>), dim3(grid2), dim3(kStBlock), l3, c->stream, g, (const uint32_t*)b.sidx,
                           (const T*)sval, b.didx, dval);
        constexpr size_t l6 = kStBin + kStBin / sizeof(T) / 8;
        EDPP_HIP(c, hipFuncSetAttribute((const void*)k_st_bins<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l6));
        hipLaunchKernelGGL((k_st_bins<T>), dim3((unsigned)std::min<int64_t>(nbins, (int64_t)std::max(c->cus, 1) * 4)),
                           dim3(kStBinBlock), l6, c->stream, g, nbins, (const uint32_t*)b.didx, (const T*)dval, out);
    } else {
        constexpr size_t l5 = st_return_lds<T>();
        EDPP_HIP(c, hipFuncSetAttribute((const void*)k_st_return<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)l5));
        hipLaunchKernelGGL((k_st_gather<T>), dim3((unsigned)ceil_div(g.n, (int64_t)kStPart<T>)), dim3(256), 0, c->stream, in,
                           g, (const uint32_t*)b.sidx, sval);
        hipLaunchKernelGGL((k_st_return<T>), dim3(grid), dim3(kStBlock), l5, c->stream, out, g, (const T*)sval,
                           (const uint16_t*)b.slot);
    }
    EDPP_HIP(c, hipGetLastError());
    return EDPP_OK;
}

int st_ceil_lg(int64_t x) {
    int l = 0;
    while ((1ll << l) < x) ++l;
    return l;
}

}  // namespace

template <class T>
int launch_gs_staged(edpp_ctx* c, const T* in, T* out, const int32_t* idx, int64_t n, bool scatter, bool* ran) {
    *ran = false;
    if (!gs_staged_applies(in, out, idx, n, (int)sizeof(T), scatter)) return EDPP_OK;
    // A graph keeps the pointers it was captured with, and may be replayed when
    // the workspace has been given back for a larger one, or beside other work
    // on the context's gate words.  So a stream under capture takes the direct
    // passes, of which a single one holds nothing but the caller's buffers.
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c->stream, &cap) != hipSuccess) {
        (void)hipGetLastError();  // some other capture forbids the question
        return EDPP_OK;
    }
    if (cap != hipStreamCaptureStatusNone) return EDPP_OK;
    constexpr int64_t S = kStTile<T>;
    StGeom g = {};
    g.n = n;
    g.chunks = ceil_div(n, (int64_t)kStChunk);
    g.tiles = ceil_div(n, S);
    g.group = st_group(g.tiles);
    g.groups = ceil_div(g.tiles, (int64_t)g.group);
    g.xcds = c->xcds;
    g.near = (uint32_t)(kStWindow / (int64_t)sizeof(T));
    int64_t nbins = 0;
    if (!scatter) {
        g.shift = st_ceil_lg(kStWindow / (int64_t)sizeof(T));
    } else {  // 128 to 256 windows of 64 or 128 bins
        g.sub_shift = st_ceil_lg(kStBin / (int64_t)sizeof(T));
        nbins = ceil_div(n, 1ll << g.sub_shift);
        g.lg_subs = st_ceil_lg(nbins) / 2;
        g.shift = g.sub_shift + g.lg_subs;
    }
    g.W = (int)ceil_div(n, 1ll << g.shift);
    g.WP = (g.W + 1) & ~1;
    const int64_t tiles2 = scatter ? g.tiles + g.W : 0;
    // workspace, in this order
    size_t at = 0;
    auto take = [&at](size_t bytes) {
        const size_t p = at;
        at += (bytes + 255) & ~(size_t)255;
        return p;
    };
    const size_t o_done = take((size_t)(g.tiles * S / kStChunk)), o_count = take((size_t)g.chunks * g.WP * 2),
                 o_rows = take((size_t)g.tiles * g.WP * 4), o_gsum = take((size_t)g.groups * g.WP * 4), o_total = take((size_t)g.WP * 4), o_open = take(4), o_base = take(((size_t)g.WP + 1) * 4),
                 o_tile2 = take(((size_t)g.WP + 1) * 4), o_win2 = take((size_t)tiles2 * 2), o_rows2 = take(((size_t)tiles2 << g.lg_subs) * 4),
                 o_bins = take(((size_t)g.W << g.lg_subs) * 4), o_sidx = take((size_t)n * 4),
                 o_sval = !scatter && sizeof(T) == 4 ? o_sidx : take((size_t)n * sizeof(T)), o_didx = take(scatter ? (size_t)n * 4 : 0),
                 o_dval = take(scatter ? (size_t)n * sizeof(T) : 0), o_slot = take(scatter ? 0 : (size_t)g.tiles * S * 2),
                 o_probe = take(scatter ? 0 : (size_t)kStProbes * 8);
    void* w;
    int rc = ws_try_reserve(c, at, &w);
    if (rc || !w) return rc;  // the direct passes need no copies
    char* p = static_cast<char*>(w);
    auto u32 = [p](size_t o) { return reinterpret_cast<uint32_t*>(p + o); };
    g.done = reinterpret_cast<uint8_t*>(p + o_done);
    g.count = reinterpret_cast<uint16_t*>(p + o_count);
    g.rows = u32(o_rows);
    g.gsum = u32(o_gsum);
    g.total = u32(o_total);
    g.open = u32(o_open);
    g.probe = u32(o_probe);
    g.base = u32(o_base);
    if (scatter) {
        g.tile2 = u32(o_tile2);
        g.win2 = reinterpret_cast<uint16_t*>(p + o_win2);
        g.rows2 = u32(o_rows2);
        g.bins = u32(o_bins);
    }
    const StBufs b = {u32(o_sidx), u32(o_didx), p + o_sval, p + o_dval, reinterpret_cast<uint16_t*>(p + o_slot)};
    g.gate = c->gs_gate;
    *ran = true;
    return scatter ? run_staged<T, true>(c, in, out, idx, g, b, nbins)
                   : run_staged<T, false>(c, in, out, idx, g, b, 0);
}

// A call whose chunks are all done directly pays for the kernels around the
// first one (the probe 8 us, those that return at once 2 to 8 us each), but
// not for the later passes of the direct schedule.  us, direct schedule / by
// this path:
//                     random permutation   4096-element blocks   two halves
//   gather  4 B  2^26     1281 /  666          112 / 135           97 / 123
//   gather  4 B  2^27     2564 / 1337          289 / 317          257 / 285
//   gather  4 B  2^28     5455 / 2766          562 / 606          518 / 551
//   scatter 4 B  2^26     1241 /  682          127 / 137          218 / 143
//   scatter 4 B  2^27     2287 / 1367          344 / 332          817 / 317
//   scatter 4 B  2^28     4481 / 2800          686 / 649         1610 / 626
//   gather  8 B  2^24      329 /  221           44 /  61           43 /  62
//   gather  8 B  2^25      663 /  455           84 / 106           80 / 103
//   gather  8 B  2^26     1317 /  890          226 / 258          222 / 247
//   gather  8 B  2^27     2931 / 1832          451 / 495          462 / 495
//   scatter 8 B  2^25      586 /  517          109 / 123          179 / 127
//   scatter 8 B  2^26     1400 / 1014          287 / 289          623 / 294
//   scatter 8 B  2^27     2800 / 2087          571 / 566         1218 / 560
// So calls start at 512 MiB, from where a local gather and scatter together
// take no longer than by the direct schedule or little more (4 B, 2^26: 272
// against 239 us, 2^27: 649 and 634); a direct gather of smaller tables loses
// a fifth or more where its indices are in streams.  The upper bound is 1024
// windows, and byte offsets of 31 bits.
bool gs_staged_applies(const void* in, const void* out, const int32_t* idx, int64_t n, int elem_bytes, bool scatter) {
    const int64_t bytes = n * elem_bytes;
    const int64_t least = 512ll << 20;
    return aligned16(in) && aligned16(out) && aligned16(idx) && bytes >= least && bytes <= kStWindow * kStMaxWindows &&
           bytes < (1ll << 31);
}

template int launch_gs_staged<uint32_t>(edpp_ctx*, const uint32_t*, uint32_t*, const int32_t*, int64_t, bool, bool*);
template int launch_gs_staged<uint64_t>(edpp_ctx*, const uint64_t*, uint64_t*, const int32_t*, int64_t, bool, bool*);

}  // namespace edpp
