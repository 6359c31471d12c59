// gather.hip — multi-pass gather and scatter.
//
// Reference: opencl/primitives/gatherImpl.cpp:7-55, scatterImpl.cpp:9-54
// (host pass loop), opencl/kernels/gather_kernel.cl:6-19,
// scatter_kernel.cl:6-21 (kernels).  Semantics kept: pass k of P handles the
// indices inside [k*ceil(n/P), (k+1)*ceil(n/P)), so the random-side working
// set of one pass is n/P elements and can stay in L2 / Infinity Cache while
// the sequential index stream is re-read every pass.
//
// MI355X layout: each lane owns U groups of 2 or 4 consecutive positions; the
// index (and, for scatter, value) groups are read as vectors with
// non-temporal hints so the streaming side does not evict the random side.
#include <algorithm>
#include "ctx.hpp"
#include "device.hpp"

namespace edpp {

// A lane's step is a group of consecutive positions, and a workgroup's 1024
// positions.  Scatters: 256 lanes of 4.  Gathers: 256 lanes of 4 4-byte values
// or 512 of 2 8-byte ones, so that the CU has 32 waves beside LDS windows of 32
// KiB, not 16, and a wave's 16-byte vectors are contiguous: local, 2^21 and
// 2^22 positions, 6.2 and 11.2 us, with 256 lanes of 4 9.1 and 18.2; random
// ones the same; 8 to 64 interleaved streams a power of two apart 5 to 20 %
// longer (8 streams, 2^22: 15.4 and 12.5), as a wave's loads then touch twice
// as many.  (512 lanes of 4: local 7.6 and 16.1.  Scatters gained a tenth where they are local, but random
// ones of 2^24 took 340 us instead of 303.)
template <class T, bool SC>
constexpr int kGsE = SC ? 4 : 16 / (int)sizeof(T);
template <class T, bool SC>
constexpr int kGsBlock = 1024 / kGsE<T, SC>;

// group g of E consecutive elements, by vectors of 16 bytes or less
template <class T, int E>
__device__ __forceinline__ void load_group(const T* p, int64_t g, T (&v)[E]) {
    constexpr int N = 16 / (int)sizeof(T) < E ? 16 / (int)sizeof(T) : E;
    typedef T vec __attribute__((ext_vector_type(N)));
    #pragma unroll
    for (int h = 0; h < E / N; ++h) {
        const vec y = ld_stream(reinterpret_cast<const vec*>(p) + g * (E / N) + h);
        #pragma unroll
        for (int k = 0; k < N; ++k) v[h * N + k] = y[k];
    }
}
template <class T, int E>
__device__ __forceinline__ void store_group(T* p, int64_t g, const T (&v)[E]) {
    static_assert(sizeof(T) * E == 16);
    typedef T vec __attribute__((ext_vector_type(E)));
    vec y;
    #pragma unroll
    for (int k = 0; k < E; ++k) y[k] = v[k];
    st_stream(y, reinterpret_cast<vec*>(p) + g);
}

// Window staging.  A workgroup's chunk is 1024*U consecutive positions.  When
// the in-slice indices of the chunk fall inside a window of kGsWin elements
// (a block-local permutation: shuffled 4096-element blocks, shuffled inside),
// the random side goes through LDS: a gather loads the window with
// consecutive loads and reads its values from LDS; a scatter writes its values
// into the window and stores the covered positions as consecutive runs, so
// the lines of the block leave whole instead of as 4-byte pieces.  Otherwise
// the random side is addressed directly.
//
// With several passes the window test runs in the first pass over all of
// the chunk's indices in [0, n); a chunk that fits is done there at once
// (each position is still written exactly once) and marked in done[], and the
// later passes skip it without reading its indices.  A block-local
// permutation so costs one pass whatever the pass count.
constexpr int kGsWin = 4096;
enum GsPhase { kGsOnly = 0, kGsFirst = 1, kGsLater = 2 };

// Smallest and largest index in [0, nall) of the workgroup's chunk (lo > hi
// when there is none), the same in every lane.  Ends with a barrier.
template <int U, int E, int BLOCK>
__device__ __forceinline__ void chunk_window(const uint32_t (&pos)[U][E], uint32_t nall, uint32_t* wlo, uint32_t* whi,
                                             uint32_t& lo, uint32_t& hi) {
    lo = 0xFFFFFFFFu;
    hi = 0;
    #pragma unroll
    for (int u = 0; u < U; ++u)
        #pragma unroll
        for (int k = 0; k < E; ++k)
            if (pos[u][k] < nall) {
                lo = std::min(lo, pos[u][k]);
                hi = std::max(hi, pos[u][k]);
            }
    #pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        lo = std::min(lo, (uint32_t)__shfl_xor((int)lo, o));
        hi = std::max(hi, (uint32_t)__shfl_xor((int)hi, o));
    }
    const int w = threadIdx.x / kWave;
    if (lane_id() == 0) {
        wlo[w] = lo;
        whi[w] = hi;
    }
    __syncthreads();
    #pragma unroll
    for (int q = 0; q < BLOCK / kWave; ++q) {
        lo = std::min(lo, wlo[q]);
        hi = std::max(hi, whi[q]);
    }
}

// out[i] = in[idx[i]] for idx[i] in [from, from+span).  The host clamps
// from+span to n, so an index outside [0,n) is skipped instead of read.
// Chunks of the first pass (kGsBlock*UF groups each) that its window
// path finished, from done[]: skip[u] for the workgroup's u-th slice of
// kGsBlock groups, the same in the whole workgroup.  Returns whether
// every slice is skipped.  A later pass may run with more vectors per lane
// (U > UF) than the first.
// ufs = log2 of the first pass's vectors per lane, which divides U; nchunk =
// the first pass's chunks (flags).  Shifts only: the test runs in every
// workgroup of every later pass.
template <int U, int BLOCK>
__device__ __forceinline__ bool later_skips(const uint8_t* __restrict__ done, int64_t ngrp, int ufs, uint32_t nchunk,
                                            bool (&skip)[U]) {
    // the workgroup's slices belong to the U >> ufs consecutive first-pass
    // chunks from blockIdx.x * (U >> ufs), one flag each
    const int per = U >> ufs;
    const uint32_t c0 = blockIdx.x * (uint32_t)per;
    uint32_t mask = 0;
    for (int f = 0; f < per; ++f)
        if (c0 + f < nchunk && done[c0 + f]) mask |= 1u << f;
    bool all = true;
    #pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t slice = (int64_t)blockIdx.x * U + u;  // its first group: slice * BLOCK
        skip[u] = slice * BLOCK >= ngrp || ((mask >> (u >> ufs)) & 1u) != 0;
        all = all && skip[u];
    }
    return all;
}

template <class T, int U, bool RNT>
__global__ __launch_bounds__((kGsBlock<T, false>)) void k_gather(const T* __restrict__ in, T* __restrict__ out,
                                                     const int32_t* __restrict__ idx, int64_t ngrp, uint32_t from,
                                                     uint32_t span, uint32_t nall, uint8_t* __restrict__ done,
                                                     int phase, int ufs, uint32_t nchunk) {
    constexpr int E = kGsE<T, false>, BLOCK = kGsBlock<T, false>;
    __shared__ T win[kGsWin];
    __shared__ uint32_t wlo[BLOCK / kWave], whi[BLOCK / kWave];
    // a gather's later passes use the first pass's vectors per lane: one flag
    // per workgroup
    (void)ufs;
    (void)nchunk;
    if (phase == kGsLater && done[blockIdx.x]) return;  // the same in the whole workgroup
    const int64_t g0 = (int64_t)blockIdx.x * BLOCK * U + threadIdx.x;
    uint32_t pos[U][E];
    #pragma unroll
    for (int u = 0; u < U; ++u) {
        int64_t g = g0 + (int64_t)u * BLOCK;
        if (g < ngrp) {
            load_group<uint32_t, E>(reinterpret_cast<const uint32_t*>(idx), g, pos[u]);
        } else {
            #pragma unroll
            for (int k = 0; k < E; ++k) pos[u][k] = nall;  // out of range
        }
    }
    T val[U][E];
    bool window = false;
    if (phase != kGsLater) {
        uint32_t lo, hi;
        chunk_window<U, E, BLOCK>(pos, nall, wlo, whi, lo, hi);
        window = lo <= hi && hi - lo < (uint32_t)kGsWin;  // the same in the whole workgroup
        if (phase == kGsFirst && threadIdx.x == 0) done[blockIdx.x] = window ? 1 : 0;
        if (window) {
            for (uint32_t o = threadIdx.x; o <= hi - lo; o += BLOCK) win[o] = in[lo + o];
            __syncthreads();
            #pragma unroll
            for (int u = 0; u < U; ++u)
                #pragma unroll
                for (int k = 0; k < E; ++k) val[u][k] = pos[u][k] < nall ? win[pos[u][k] - lo] : T(0);
            // every index of the chunk is done: the slice of this pass is all of [0, n)
            from = 0;
            span = nall;
        }
    }
    if (!window) {
        #pragma unroll
        for (int u = 0; u < U; ++u)
            #pragma unroll
            for (int k = 0; k < E; ++k)
                val[u][k] = (pos[u][k] - from < span) ? (RNT ? ld_stream(in + pos[u][k]) : in[pos[u][k]]) : T(0);
    }
    #pragma unroll
    for (int u = 0; u < U; ++u) {
        int64_t g = g0 + (int64_t)u * BLOCK;
        if (g < ngrp) {
            bool all = true;
            #pragma unroll
            for (int k = 0; k < E; ++k) all = all && (pos[u][k] - from < span);
            if (all) {
                store_group<T, E>(out, g, val[u]);
            } else {
                #pragma unroll
                for (int k = 0; k < E; ++k)
                    if (pos[u][k] - from < span) out[E * g + k] = val[u][k];
            }
        }
    }
}

// out[idx[i]] = in[i] for idx[i] in [from, from+span)
template <class T, int U, bool RNT>
__global__ __launch_bounds__((kGsBlock<T, true>)) void k_scatter(const T* __restrict__ in, T* __restrict__ out,
                                                      const int32_t* __restrict__ idx, int64_t ngrp, uint32_t from,
                                                      uint32_t span, uint32_t nall, uint8_t* __restrict__ done,
                                                      int phase, int ufs, uint32_t nchunk) {
    constexpr int E = kGsE<T, true>, BLOCK = kGsBlock<T, true>;
    __shared__ T win[kGsWin];
    __shared__ uint32_t cov[kGsWin / 32];  // positions of the window this chunk writes
    __shared__ uint32_t wlo[BLOCK / kWave], whi[BLOCK / kWave];
    bool skip[U] = {};
    if (phase == kGsLater && later_skips<U, BLOCK>(done, ngrp, ufs, nchunk, skip)) return;
    for (int i = threadIdx.x; i < kGsWin / 32; i += BLOCK) cov[i] = 0;
    const int64_t g0 = (int64_t)blockIdx.x * BLOCK * U + threadIdx.x;
    uint32_t pos[U][E];
    T val[U][E];
    #pragma unroll
    for (int u = 0; u < U; ++u) {
        int64_t g = g0 + (int64_t)u * BLOCK;
        if (g < ngrp && !skip[u]) {
            load_group<uint32_t, E>(reinterpret_cast<const uint32_t*>(idx), g, pos[u]);
            load_group<T, E>(in, g, val[u]);
        } else {
            #pragma unroll
            for (int k = 0; k < E; ++k) { pos[u][k] = nall; val[u][k] = 0; }
        }
    }
    bool window = false;
    if (phase != kGsLater) {
        uint32_t lo, hi;
        chunk_window<U, E, BLOCK>(pos, nall, wlo, whi, lo, hi);  // its barrier also orders the cov clearing
        window = lo <= hi && hi - lo < (uint32_t)kGsWin;  // the same in the whole workgroup
        if (phase == kGsFirst && threadIdx.x == 0) done[blockIdx.x] = window ? 1 : 0;
        if (window) {
            #pragma unroll
            for (int u = 0; u < U; ++u)
                #pragma unroll
                for (int k = 0; k < E; ++k)
                    if (pos[u][k] < nall) {
                        const uint32_t o = pos[u][k] - lo;
                        win[o] = val[u][k];
                        atomicOr(cov + (o >> 5), 1u << (o & 31));
                    }
            __syncthreads();
            for (uint32_t o = threadIdx.x; o <= hi - lo; o += BLOCK)
                if ((cov[o >> 5] >> (o & 31)) & 1u) out[lo + o] = win[o];
        }
    }
    if (!window) {
        #pragma unroll
        for (int u = 0; u < U; ++u)
            #pragma unroll
            for (int k = 0; k < E; ++k)
                if (pos[u][k] - from < span) {
                    if (RNT) st_stream(val[u][k], out + pos[u][k]);
                    else out[pos[u][k]] = val[u][k];
                }
    }
}

// elements [lo, n): scalar tail and the path for unaligned pointers
template <class T>
__global__ void k_gs_scalar(const T* in, T* out, const int32_t* idx, int64_t lo, int64_t n, uint32_t from,
                            uint32_t span, bool scatter) {
    for (int64_t i = lo + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        uint32_t p = (uint32_t)idx[i];
        if (p - from < span) {
            if (scatter) out[p] = in[i];
            else out[i] = in[p];
        }
    }
}

struct GsPass {
    uint32_t from, span, nall;
    uint8_t* done;  // one flag per workgroup chunk, written by the first of several passes
    int phase;
    int ufs;          // log2 of the first pass's groups per lane (one done flag per 1024 << ufs positions)
    uint32_t nchunk;  // done flags (workgroups of the first pass)
};

template <class T, int U, bool RNT>
static void launch_gs_kernel(edpp_ctx* c, const T* in, T* out, const int32_t* idx, int64_t ngrp, const GsPass& q,
                             bool scatter) {
    const int block = scatter ? kGsBlock<T, true> : kGsBlock<T, false>;
    const unsigned grid = (unsigned)ceil_div(ngrp, (int64_t)block * U);
    hipLaunchKernelGGL((scatter ? k_scatter<T, U, RNT> : k_gather<T, U, RNT>), dim3(grid), dim3(block), 0, c->stream, in,
                       out, idx, ngrp, q.from, q.span, q.nall, q.done, q.phase, q.ufs, q.nchunk);
}

template <class T, bool RNT>
static void dispatch_unroll(edpp_ctx* c, int u, const T* in, T* out, const int32_t* idx, int64_t ngrp,
                            const GsPass& q, bool scatter) {
    switch (u) {
        case 1: launch_gs_kernel<T, 1, RNT>(c, in, out, idx, ngrp, q, scatter); break;
        case 2: launch_gs_kernel<T, 2, RNT>(c, in, out, idx, ngrp, q, scatter); break;
        case 8: launch_gs_kernel<T, 8, RNT>(c, in, out, idx, ngrp, q, scatter); break;
        default: launch_gs_kernel<T, 4, RNT>(c, in, out, idx, ngrp, q, scatter); break;
    }
}

template <class T>
int launch_gather(edpp_ctx* c, const T* in, T* out, const int32_t* idx, int64_t n, int passes, bool scatter) {
    if (n == 0) return EDPP_OK;
    if (passes == 0) passes = default_passes(c, n, (int)sizeof(T), scatter);
    if (passes < 1 || passes > n) passes = passes < 1 ? 1 : (int)n;
    const bool vec = aligned16(in) && aligned16(out) && aligned16(idx);
    const int e = scatter ? kGsE<T, true> : kGsE<T, false>, block = 1024 / e;
    const int64_t ngrp = vec ? n / e : 0;
    const int64_t len = ceil_div(n, passes);  // gatherImpl.cpp:37
    uint8_t* done = nullptr;
    if (ngrp && passes > 1) {
        const int64_t grid = ceil_div(ngrp, (int64_t)block * c->tune.gs_unroll);
        void* w;
        int rc = ws_reserve(c, (size_t)grid, &w);
        if (rc) return rc;
        done = static_cast<uint8_t*>(w);
    }
    for (int p = 0; p < passes; ++p) {
        const int64_t lo = (int64_t)p * len;
        if (lo >= n) break;
        GsPass q;
        q.from = (uint32_t)lo;
        q.span = (uint32_t)(lo + len <= n ? len : n - lo);
        q.nall = (uint32_t)n;
        q.done = done;
        q.phase = passes == 1 ? kGsOnly : (p == 0 ? kGsFirst : kGsLater);
        const int uf = c->tune.gs_unroll;  // 1, 2, 4 or 8
        q.ufs = uf == 1 ? 0 : uf == 2 ? 1 : uf == 4 ? 2 : 3;
        q.nchunk = (uint32_t)ceil_div(ngrp, (int64_t)block * uf);
        const uint32_t from = q.from, span = q.span;
        // scatter passes after the first skip the window test, so for 4-byte
        // values they take 8 index vectors per lane: half the workgroups
        // re-reading the index and values (2^28, random, 4 passes: 4.51
        // against 4.95 ms; gathers measured no steady gain)
        const int u = (q.phase == kGsLater && scatter && sizeof(T) == 4) ? std::max(8, uf) : uf;
        if (ngrp) {
            if (c->tune.gs_random_nt > 0)
                dispatch_unroll<T, true>(c, u, in, out, idx, ngrp, q, scatter);
            else
                dispatch_unroll<T, false>(c, u, in, out, idx, ngrp, q, scatter);
        }
        if (ngrp * e < n) {
            int64_t rest = n - ngrp * e;
            unsigned g = (unsigned)(rest < 256 * 4096 ? ceil_div(rest, 256) : 4096);
            hipLaunchKernelGGL((k_gs_scalar<T>), dim3(g), dim3(256), 0, c->stream, in, out, idx, ngrp * e, n, from,
                               span, scatter);
        }
    }
    EDPP_HIP(c, hipGetLastError());
    return EDPP_OK;
}

template int launch_gather<uint32_t>(edpp_ctx*, const uint32_t*, uint32_t*, const int32_t*, int64_t, int, bool);
template int launch_gather<uint64_t>(edpp_ctx*, const uint64_t*, uint64_t*, const int32_t*, int64_t, int, bool);

}  // namespace edpp
