// join.hip — partitioned hash join (count of equal-key pairs) on the stable
// split.
//
// Reference: obsolete/OpenCL/phjImpl.cpp:14-66 (partition R and S with
// WG_split into 2^13 buckets, then one workgroup per bucket pair builds an LDS
// hash table of one side and probes it with the other,
// obsolete/OpenCL/hj_partitioned_kernel.cl:7-115) and its count-only result
// (phjImpl.cpp:13 "only count the number of outputs").  The count is
//   sum over keys k of |{i: R[i] == k}| * |{j: S[j] == k}|.
// Here the keys are replaced by a bijective mix of their bits (mix32), so that
// the partitions stay balanced for structured keys; equal keys keep equal
// mixes.  The partitioning mixes each key as it loads it, so the mixed keys
// are never written and read back by a pass of their own.
//
// A count does not depend on the order inside a partition, so relations of up
// to 2^24 keys (the smaller one) are partitioned by the mix's top bits into at
// most 1024 windows in one pass, both in the same launches (k_jn_hist,
// k_st_groups, k_st_totals, k_jn_split); longer ones by the stable split's two passes.
// The partition pairs are then joined by persistent workgroups with a hash
// table in LDS: 64-bit slots and 4096 build keys per partition (k_join_probe),
// or, where partitions are fewer, 16 384 build keys in bucket order or in
// 32-bit slots (k_jn_probe).  Every key is valid (no sentinel value, unlike the reference's
// -1), and any skew ends, at the cost of re-probing.
#include <algorithm>
#include "ctx.hpp"
#include "device.hpp"
#include "split_tile.hpp"
#include "window_tile.hpp"

namespace edpp {

namespace {

constexpr int kJoinBlock = 1024;
constexpr int kJoinSlots = 16384;  // 64-bit LDS slots (128 KiB): (count << 32) | key; count 0 = empty
constexpr int kJoinChunk = kJoinSlots / 2;  // build keys per table fill
constexpr int kJoinTargetBuild = 4096;
constexpr int kJoinPre = kJoinChunk / kJoinBlock;  // keys per lane per side held in registers (8)
// Partition bits at most: the split runs up to 16 bucket bits as two stable
// passes, so relations up to 2^28 keys keep about kJoinTargetBuild build keys
// per partition and one table fill each.
constexpr int kJoinMaxBits = 16;

__global__ void k_join_zero(unsigned long long* p) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *p = 0ull;
}

// Slots are probed from the mixed key's bits above the partition bits.
__device__ __forceinline__ uint32_t join_slot(uint32_t hk, int pbits) {
    return (pbits >= 32 ? 0u : (hk >> pbits)) & (uint32_t)(kJoinSlots - 1);
}

// A claim is tried first: on an empty slot (most of them, at a load factor
// of at most 1/2) it is the only LDS operation; a failed claim returns the
// slot's word, whose key never changes once set.  Returns the slot this
// call claimed, or kNoClaim when the key was counted into a slot that
// another call had claimed.
constexpr uint32_t kNoClaim = 0xFFFFFFFFu;
__device__ __forceinline__ uint32_t join_insert(uint64_t* table, uint32_t hk, int pbits) {
    uint32_t h = join_slot(hk, pbits);
    while (true) {
        uint64_t w = 0;  // empty: claim it for this key with count 1
        if (__hip_atomic_compare_exchange_strong(table + h, &w, (1ull << 32) | hk, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP))
            return h;
        if ((uint32_t)w == hk) {
            __hip_atomic_fetch_add(table + h, 1ull << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            return kNoClaim;
        }
        h = (h + 1) & (uint32_t)(kJoinSlots - 1);
    }
}

__device__ __forceinline__ uint32_t join_lookup(const uint64_t* table, uint32_t hk, int pbits) {
    uint32_t h = join_slot(hk, pbits);
    while (true) {
        const uint64_t w = table[h];
        if ((w >> 32) == 0) return 0;
        if ((uint32_t)w == hk) return (uint32_t)(w >> 32);
        h = (h + 1) & (uint32_t)(kJoinSlots - 1);
    }
}

// Rows of partition pair b: R rows [rs[b], rs[b+1]) and S rows [ss[b],
// ss[b+1]) of the partitioned mixed keys, the smaller side built into the
// table.  The offsets are clamped to the relations: a split whose device
// wait timed out (reported as EDPP_ETIMEOUT) leaves offsets that must not
// steer reads.
struct JoinPair {
    const uint32_t* bkeys;
    const uint32_t* pkeys;
    int64_t b0, b1, p0, p1;
    // both sides fit the registers of one table fill (the balanced case)
    __device__ __forceinline__ bool held() const {
        return b1 > b0 && p1 > p0 && b1 - b0 <= kJoinPre * kJoinBlock && p1 - p0 <= kJoinPre * kJoinBlock;
    }
};
__device__ __forceinline__ JoinPair join_pair(int b, const uint32_t* rk, int64_t rn, const int32_t* rs,
                                              const uint32_t* sk, int64_t sn, const int32_t* ss, int B) {
    auto clamp = [](int64_t x, int64_t lo, int64_t hi) { return x < lo ? lo : (x > hi ? hi : x); };
    const int64_t r0 = clamp(rs[b], 0, rn), r1 = clamp(b + 1 < B ? rs[b + 1] : rn, r0, rn);
    const int64_t s0 = clamp(ss[b], 0, sn), s1 = clamp(b + 1 < B ? ss[b + 1] : sn, s0, sn);
    const bool build_r = (r1 - r0) <= (s1 - s0);
    JoinPair jp;
    jp.bkeys = build_r ? rk : sk;
    jp.pkeys = build_r ? sk : rk;
    jp.b0 = build_r ? r0 : s0;
    jp.b1 = build_r ? r1 : s1;
    jp.p0 = build_r ? s0 : r0;
    jp.p1 = build_r ? s1 : r1;
    return jp;
}
// lane's keys of a held pair's two sides
__device__ __forceinline__ void join_load(const JoinPair& jp, uint32_t (&bk)[kJoinPre], uint32_t (&pk)[kJoinPre]) {
    #pragma unroll
    for (int q = 0; q < kJoinPre; ++q) {
        const int64_t i = jp.b0 + threadIdx.x + (int64_t)q * kJoinBlock;
        bk[q] = i < jp.b1 ? jp.bkeys[i] : 0u;
    }
    #pragma unroll
    for (int q = 0; q < kJoinPre; ++q) {
        const int64_t i = jp.p0 + threadIdx.x + (int64_t)q * kJoinBlock;
        pk[q] = i < jp.p1 ? jp.pkeys[i] : 0u;
    }
}

// Adds the workgroup's counts to *d_count: wave sums, then one lane per wave
// through the table's first slots.
__device__ __forceinline__ void join_add_up(unsigned long long local, uint64_t* table, unsigned long long* d_count) {
    const uint64_t ws = wave_sum((uint64_t)local);
    __syncthreads();
    if (lane_id() == 0) table[threadIdx.x / kWave] = ws;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long total = 0;
        for (int q = 0; q < kJoinBlock / kWave; ++q) total += table[q];
        if (total) atomicAdd(d_count, total);
    }
}

// Persistent: workgroup g (one per CU, as its table fills the CU's LDS)
// takes partition pairs g, g + gridDim.x, ...  While a pair's table is
// cleared, filled and probed, the next pair's offsets and (when both of its
// sides fit the registers) keys are loaded, so their global latency is hidden
// behind the LDS work.  A table fill holds at most kJoinChunk distinct keys in
// kJoinSlots slots, so every probe sequence meets an empty slot and ends.
__global__ __launch_bounds__(kJoinBlock) void k_join_probe(const uint32_t* __restrict__ rk, int64_t rn,
                                                           const int32_t* __restrict__ rs,
                                                           const uint32_t* __restrict__ sk, int64_t sn,
                                                           const int32_t* __restrict__ ss, int B, int pbits,
                                                           unsigned long long* d_count) {
    extern __shared__ uint64_t table[];  // kJoinSlots
    unsigned long long local = 0;
    int b = blockIdx.x;
    JoinPair cur = join_pair(b, rk, rn, rs, sk, sn, ss, B);
    uint32_t bk[kJoinPre], pk[kJoinPre];
    if (cur.held()) join_load(cur, bk, pk);
    // after a held pair the only nonzero slots are the ones its lanes
    // claimed (recorded in claimed[]): the next held pair clears just those
    bool sparse = false;
    uint32_t claimed[kJoinPre];
    for (; b < B; b += gridDim.x) {
        const int nb = b + (int)gridDim.x;
        JoinPair nxt = cur;
        if (nb < B) nxt = join_pair(nb, rk, rn, rs, sk, sn, ss, B);
        uint32_t nbk[kJoinPre], npk[kJoinPre];
        __syncthreads();  // the previous pair's lookups are done before the table is cleared
        if (cur.held()) {
            if (sparse) {
                #pragma unroll
                for (int q = 0; q < kJoinPre; ++q)
                    if (claimed[q] != kNoClaim) table[claimed[q]] = 0ull;
            } else {
                for (int i = threadIdx.x; i < kJoinSlots; i += kJoinBlock) table[i] = 0ull;
            }
            if (nb < B && nxt.held()) join_load(nxt, nbk, npk);
            __syncthreads();
            #pragma unroll
            for (int q = 0; q < kJoinPre; ++q)
                claimed[q] = cur.b0 + threadIdx.x + (int64_t)q * kJoinBlock < cur.b1 ? join_insert(table, bk[q], pbits)
                                                                                     : kNoClaim;
            sparse = true;
            __syncthreads();
            #pragma unroll
            for (int q = 0; q < kJoinPre; ++q)
                if (cur.p0 + threadIdx.x + (int64_t)q * kJoinBlock < cur.p1)
                    local += join_lookup(table, pk[q], pbits);
        } else {
            if (nb < B && nxt.held()) join_load(nxt, nbk, npk);
            if (cur.b1 > cur.b0 && cur.p1 > cur.p0) {
                sparse = false;  // the chunk fills leave slots no lane recorded
                for (int64_t c0 = cur.b0; c0 < cur.b1; c0 += kJoinChunk) {
                    const int64_t c1 = std::min<int64_t>(c0 + kJoinChunk, cur.b1);
                    for (int i = threadIdx.x; i < kJoinSlots; i += kJoinBlock) table[i] = 0ull;
                    __syncthreads();
                    for (int64_t i = c0 + threadIdx.x; i < c1; i += kJoinBlock)
                        join_insert(table, cur.bkeys[i], pbits);
                    __syncthreads();
                    for (int64_t i = cur.p0 + threadIdx.x; i < cur.p1; i += kJoinBlock)
                        local += join_lookup(table, cur.pkeys[i], pbits);
                    __syncthreads();
                }
            }
        }
        cur = nxt;
        #pragma unroll
        for (int q = 0; q < kJoinPre; ++q) {
            bk[q] = nbk[q];
            pk[q] = npk[q];
        }
    }
    join_add_up(local, table, d_count);
}

// ------------------------------------------------------------- one-pass partition
constexpr int kJnEpl = 32;                        // keys per lane of a tile
constexpr int kJnTile = kStBlock * kJnEpl;        // 16,384 keys
constexpr int kJnCh = kJnTile / kStChunk;
constexpr int kJnMaxBits = 10;                    // at most kStMaxWindows partitions
struct JnRel {
    const uint32_t* keys;
    uint32_t* part;
    StGeom g;
};

// chunk counts of both relations (grid.y); the count is cleared here
__global__ __launch_bounds__(256) void k_jn_hist(JnRel r0, JnRel r1, unsigned long long* d_count) {
    __shared__ uint32_t cnt[kStBuckets];
    const JnRel& r = blockIdx.y ? r1 : r0;
    const StGeom& g = r.g;
    const int t = threadIdx.x;
    if (blockIdx.x == 0 && blockIdx.y == 0 && t == 0) *d_count = 0ull;
    if ((int64_t)blockIdx.x >= g.chunks) return;
    const int64_t v0 = (int64_t)blockIdx.x * (kStChunk / 4) + t;
    uint32_t x[16];
    #pragma unroll
    for (int u = 0; u < 4; ++u) st_load<uint32_t, 4>(r.keys, v0 + u * 256, g.n, 0u, x + 4 * u);
    const int cl = st_copies_lg(g.W);
    for (int i = t; i < (g.WP << cl); i += 256) cnt[i] = 0;
    __syncthreads();
    const uint32_t copy = t & ((1u << cl) - 1u);
    #pragma unroll
    for (int e = 0; e < 16; ++e)
        if (4 * (v0 + e / 4 * 256) + e % 4 < g.n)
            __hip_atomic_fetch_add(cnt + ((mix32(x[e]) >> g.shift) << cl) + copy, 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    uint32_t* row = reinterpret_cast<uint32_t*>(g.count + (int64_t)blockIdx.x * g.WP);
    for (int i = t; i < g.WP / 2; i += 256) {
        uint32_t a = 0, b = 0;
        for (int c = 0; c < (1 << cl); ++c) {
            a += cnt[((2 * i) << cl) + c];
            b += cnt[((2 * i + 1) << cl) + c];
        }
        row[i] = a | (b << 16);
    }
}

constexpr size_t kJnSplitLds = (size_t)kJnTile * 4 + 8 * kStBuckets;
// mixed keys of one tile to their partitions
__global__ __launch_bounds__(kStBlock, kStBlock / 128) void k_jn_split(JnRel r0, JnRel r1) {
    extern __shared__ uint32_t buf[];  // [tile], then counts and offsets
    uint32_t* cnt = buf + kJnTile;
    uint32_t* off = cnt + kStBuckets;
    __shared__ uint32_t wtmp[kStBlock / kWave];
    const JnRel& r = blockIdx.y ? r1 : r0;
    const StGeom& g = r.g;
    if ((int64_t)blockIdx.x >= g.tiles) return;
    const int64_t tile = st_order(blockIdx.x, (uint32_t)g.tiles, g.xcds);
    const uint32_t tid = threadIdx.x;
    if (blockIdx.x == 0) st_keep_bases<kJnCh>(g, tid, wtmp, off);
    const int cl = st_copies_lg(g.W);
    const int left = (int)std::min<int64_t>(g.n - tile * kJnTile, kJnTile) - (int)tid * 4;
    uint32_t m;
    {
        uint32_t x[kJnEpl], at[kJnEpl / 2];
        if (left + (int)tid * 4 == kJnTile) {
            #pragma unroll
            for (int u = 0; u < kJnEpl / 4; ++u) {
                const v4u32 v = ld_stream(reinterpret_cast<const v4u32*>(r.keys) + tile * (kJnTile / 4) + u * kStBlock + tid);
                #pragma unroll
                for (int k = 0; k < 4; ++k) x[4 * u + k] = v[k];
            }
        } else {
            const __amdgpu_buffer_rsrc_t rs = buf_rsrc(r.keys + tile * kJnTile, g.n - tile * kJnTile);
            #pragma unroll
            for (int e = 0; e < kJnEpl; ++e) x[e] = buf_load<uint32_t>(rs, tid * 16, (uint32_t)(e / 4 * kStBlock * 16 + e % 4 * 4));
        }
        #pragma unroll
        for (int e = 0; e < kJnEpl; ++e) x[e] = mix32(x[e]);
        m = st_rank<kJnEpl>(
            tid, x, at,
            [&](int e, uint32_t v) { return e / 4 * kStBlock * 4 + e % 4 < left ? v >> g.shift : (uint32_t)g.W; }, g.W, cl,
            cnt, off, wtmp);
        st_place<uint32_t, kJnEpl>(buf, at, x);
    }
    __syncthreads();
    st_distances(g, tile, tid, cl, cnt, off, wtmp);
    __syncthreads();
    const BufSink<uint32_t> out = buf_sink(r.part, g.n);
    #pragma unroll
    for (int j = 0; j < kJnEpl; ++j) {
        const uint32_t i = tid + j * kStBlock;
        const uint32_t k = buf[i];
        const uint32_t d = cnt[std::min(k >> g.shift, (uint32_t)g.W - 1u)] + i;  // a slot past m holds anything
        out.put(i < m ? d : kStNone, k);
    }
}

// ------------------------------------------------------------- 32-bit slots
// Partitions of about 16,384 build keys whose mixes share their top `pbits`
// bits: a slot holds the other bits and, above them, a count of up to
// 2^pbits - 1; 0 is empty.  A key that occurs more often raises `over`, and
// the pair is joined with 64-bit slots instead.
//
// Slots lie in buckets of four, read with one 16-byte LDS load; at a load of
// 1/2 nearly every key ends in its first bucket.  2^24 x 2^24 distinct keys in
// 1024 pairs took 173 us so, VALU and LDS each busy for two fifths of it: a
// wave goes on until the last of its lanes has found its slot.  Such keys now
// take the bucket order below; these slots are for keys that repeat.
constexpr int kJnSlots = 2 * kJoinSlots;   // the same 128 KiB
constexpr int kJnBuckets = kJnSlots / 4;
constexpr int kJnPre = 18;                 // keys per lane per side held in registers: a partition of 16,384
                                           // expected keys has fewer than 18,432 but once in 10^50
__device__ __forceinline__ void jn_insert(uint32_t* table, uint32_t k, int fb, uint32_t* over) {
    const uint32_t fm = (1u << fb) - 1u, one = 1u << fb;
    const uint32_t w = one | (k & fm);
    uint32_t h = k & (uint32_t)(kJnBuckets - 1);
    while (true) {
        asm volatile("" ::: "memory");  // other lanes fill slots: read anew (a volatile read would be a flat load)
        const v4u32 v = reinterpret_cast<const v4u32*>(table)[h];
        // the key's slot, else the first empty one: slots fill in order and
        // never empty, so lanes with one key meet in one slot
        int at = -1;
        #pragma unroll
        for (int i = 3; i >= 0; --i) at = v[i] == 0u ? i : at;
        #pragma unroll
        for (int i = 0; i < 4; ++i) at = v[i] != 0u && ((v[i] ^ k) & fm) == 0 ? i : at;
        if (at < 0) {  // full
            h = (h + 1) & (uint32_t)(kJnBuckets - 1);
            continue;
        }
        uint32_t* slot = table + 4 * h + at;
        uint32_t o = 0;
        if (__hip_atomic_compare_exchange_strong(slot, &o, w, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP))
            return;
        if (((o ^ k) & fm) == 0) {
            o = __hip_atomic_fetch_add(slot, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if ((o >> fb) == (0xFFFFFFFFu >> fb)) *over = 1u;
            return;
        }
    }
}
__device__ __forceinline__ uint32_t jn_lookup(const uint32_t* table, uint32_t k, int fb) {
    const uint32_t fm = (1u << fb) - 1u;
    uint32_t h = k & (uint32_t)(kJnBuckets - 1);
    while (true) {
        const v4u32 v = reinterpret_cast<const v4u32*>(table)[h];
        uint32_t c = 0;
        #pragma unroll
        for (int i = 0; i < 4; ++i) c = v[i] != 0u && ((v[i] ^ k) & fm) == 0 ? v[i] >> fb : c;
        if (c != 0 || v[3] == 0u) return c;  // slots fill in order
        h = (h + 1) & (uint32_t)(kJnBuckets - 1);
    }
}

__device__ __forceinline__ void jn_load(const uint32_t* __restrict__ p, int64_t lo, int64_t hi, uint32_t (&x)[kJnPre]) {
    // one descriptor for the lane's keys; loads past the end read 0
    const __amdgpu_buffer_rsrc_t r = buf_rsrc(p + lo, std::min<int64_t>(hi - lo, kJnPre * kJoinBlock));
    #pragma unroll
    for (int q = 0; q < kJnPre; ++q) x[q] = buf_load<uint32_t>(r, threadIdx.x * 4, q * kJoinBlock * 4);
}

// Build keys in bucket order: bucket h's are keys[first .. first + len), from
// index[h] = first | len << 16.  An insertion is one counter atomic, with no
// claim that can fail, and a lookup reads the bucket's keys only.  2^24 x 2^24
// keys: 104 us instead of 173; one workgroup per CU, whose LDS operations and
// barriers bound it.
constexpr int kJnHeads = 16384;
// Keys that repeat make buckets long, and slots with counts are then the
// better table: a bucket of more than kJnEarly among the first keys of every
// lane, or of more than kJnDeep in the end.  2^24 x 2^24 keys that occur 4, 8
// and 16 times: 248, 243 and 242 us, and 270 to 280 where only the end tells.
constexpr int kJnFirst = 6;
constexpr uint32_t kJnEarly = 9, kJnDeep = 24;
constexpr int kJnBatch = 3;  // probes that go on together
static_assert(kJnPre % kJnBatch == 0 && kJnPre % 2 == 0);
constexpr size_t kJnLds = ((size_t)kJnHeads + kJnPre * kJoinBlock) * 4;
static_assert(kJnLds >= (size_t)kJnSlots * 4);

// index[] from counts to {first, len}.  Barriers around it.
__device__ __forceinline__ void jn_index(uint32_t* index, uint32_t* wtmp) {
    constexpr int R = kJnHeads / 4 / kJoinBlock, W = kJoinBlock / kWave;
    static_assert(R * W <= kWave);
    v4u32* v = reinterpret_cast<v4u32*>(index) + threadIdx.x;
    const int w = threadIdx.x / kWave;
    v4u32 c[R];
    uint32_t at[R];
    #pragma unroll
    for (int j = 0; j < R; ++j) c[j] = v[j * kJoinBlock];
    #pragma unroll
    for (int j = 0; j < R; ++j) {
        const uint32_t sum = c[j][0] + c[j][1] + c[j][2] + c[j][3], inc = wave_inclusive_add(sum);
        if (lane_id() == kWave - 1) wtmp[j * W + w] = inc;
        at[j] = inc - sum;
    }
    __syncthreads();
    // every wave scans all the row sums for itself
    const uint32_t sum = lane_id() < R * W ? wtmp[lane_id()] : 0u, before = wave_inclusive_add(sum) - sum;
    #pragma unroll
    for (int j = 0; j < R; ++j) {
        uint32_t f = at[j] + read_lane(before, j * W + __builtin_amdgcn_readfirstlane(w));
        v4u32 y;
        #pragma unroll
        for (int k = 0; k < 4; ++k) {
            y[k] = f | (c[j][k] << 16);
            f += c[j][k];
        }
        v[j * kJoinBlock] = y;
    }
    __syncthreads();
}

// Build keys that equal the batch's probe keys (ok: the lane has one)
__device__ __forceinline__ uint32_t jn_matches(const uint32_t* index, const uint32_t* keys,
                                               const uint32_t (&k)[kJnBatch], const bool (&ok)[kJnBatch]) {
    uint32_t at[kJnBatch], end[kJnBatch], found = 0;
    #pragma unroll
    for (int q = 0; q < kJnBatch; ++q) {
        const uint32_t x = ok[q] ? index[k[q] & (uint32_t)(kJnHeads - 1)] : 0u;
        at[q] = x & 0xFFFFu;
        end[q] = at[q] + (x >> 16);
    }
    bool more = true;
    while (more) {
        uint32_t y[kJnBatch];
        #pragma unroll
        for (int q = 0; q < kJnBatch; ++q) y[q] = at[q] < end[q] ? keys[at[q]] : ~k[q];
        more = false;
        #pragma unroll
        for (int q = 0; q < kJnBatch; ++q) {
            found += y[q] == k[q] ? 1u : 0u;
            ++at[q];
            more = more || at[q] < end[q];
        }
    }
    return found;
}

// Persistent, as k_join_probe; a side's keys of the next pair are loaded into
// the registers that this pair is done with, so the probes hide the one load
// and the next pair's counting the other.  Build keys that repeat take 32-bit
// slots with counts instead, a build side past the registers (heavy keys)
// chunked fills of 64-bit slots; a probe side past them is read on from memory.
__global__ __launch_bounds__(kJoinBlock) void k_jn_probe(const uint32_t* __restrict__ rk, int64_t rn,
                                                         const int32_t* __restrict__ rs,
                                                         const uint32_t* __restrict__ sk, int64_t sn,
                                                         const int32_t* __restrict__ ss, int B, int pbits,
                                                         unsigned long long* d_count) {
    extern __shared__ uint64_t table64[];  // kJnLds bytes
    uint32_t* table = reinterpret_cast<uint32_t*>(table64);
    uint32_t* keys = table + kJnHeads;
    v4u32* t4 = reinterpret_cast<v4u32*>(table) + threadIdx.x;
    __shared__ uint32_t over, wtmp[kWave];
    const int fb = 32 - pbits;
    unsigned long long local = 0;
    int b = blockIdx.x;
    JoinPair cur = join_pair(b, rk, rn, rs, sk, sn, ss, B);
    uint32_t bk[kJnPre], pk[kJnPre];
    jn_load(cur.bkeys, cur.b0, cur.b1, bk);
    jn_load(cur.pkeys, cur.p0, cur.p1, pk);
    for (; b < B; b += gridDim.x) {
        const int nb = b + (int)gridDim.x;
        JoinPair nxt = cur;
        if (nb < B) nxt = join_pair(nb, rk, rn, rs, sk, sn, ss, B);
        const bool any = cur.b1 > cur.b0 && cur.p1 > cur.p0;
        const bool held = any && cur.b1 - cur.b0 <= kJnPre * kJoinBlock;
        const int bn = held ? (int)(cur.b1 - cur.b0) : 0;
        const int64_t pn = cur.p1 - cur.p0;
        bool slots = false, chunks = any && !held;
        __syncthreads();  // the previous pair's lookups are done before the table is cleared
        if (held) {
            #pragma unroll
            for (int i = 0; i < kJnHeads / 4 / kJoinBlock; ++i) t4[i * kJoinBlock] = v4u32{0u, 0u, 0u, 0u};
            if (threadIdx.x == 0) over = 0u;
            __syncthreads();
            uint32_t rank[kJnPre / 2];  // two to a word
            uint32_t most = 0;
            #pragma unroll
            for (int q = 0; q < kJnPre / 2; ++q) {
                if (q == kJnFirst / 2) slots = __syncthreads_or(most >= kJnEarly);
                if (slots) continue;
                uint32_t r[2];
                #pragma unroll
                for (int h = 0; h < 2; ++h)
                    r[h] = (int)threadIdx.x + (2 * q + h) * kJoinBlock < bn
                               ? __hip_atomic_fetch_add(table + (bk[2 * q + h] & (uint32_t)(kJnHeads - 1)), 1u,
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)
                               : 0u;
                most = std::max(most, std::max(r[0], r[1]));
                rank[q] = r[0] | (r[1] << 16);
            }
            slots = __syncthreads_or(slots || most >= kJnDeep);
            if (!slots) {
                jn_index(table, wtmp);
                #pragma unroll
                for (int q = 0; q < kJnPre; ++q)
                    if ((int)threadIdx.x + q * kJoinBlock < bn)
                        keys[(table[bk[q] & (uint32_t)(kJnHeads - 1)] & 0xFFFFu) +
                             (q % 2 ? rank[q / 2] >> 16 : rank[q / 2] & 0xFFFFu)] = bk[q];
            } else {
                #pragma unroll
                for (int i = 0; i < kJnSlots / 4 / kJoinBlock; ++i) t4[i * kJoinBlock] = v4u32{0u, 0u, 0u, 0u};
                if (threadIdx.x == 0) over = 0u;
                __syncthreads();
                #pragma unroll
                for (int q = 0; q < kJnPre; ++q)
                    if ((int)threadIdx.x + q * kJoinBlock < bn) jn_insert(table, bk[q], fb, &over);
            }
        }
        if (nb < B) jn_load(nxt.bkeys, nxt.b0, nxt.b1, bk);
        if (held) {
            __syncthreads();
            chunks = over != 0u && slots;
            if (!slots) {
                #pragma unroll
                for (int q = 0; q < kJnPre; q += kJnBatch) {
                    uint32_t k[kJnBatch];
                    bool ok[kJnBatch];
                    #pragma unroll
                    for (int i = 0; i < kJnBatch; ++i) {
                        k[i] = pk[q + i];
                        ok[i] = threadIdx.x + (int64_t)(q + i) * kJoinBlock < pn;
                    }
                    local += jn_matches(table, keys, k, ok);
                }
                for (int64_t i = cur.p0 + kJnPre * kJoinBlock + threadIdx.x; i < cur.p1; i += kJnBatch * kJoinBlock) {
                    uint32_t k[kJnBatch];
                    bool ok[kJnBatch];
                    #pragma unroll
                    for (int q = 0; q < kJnBatch; ++q) {
                        ok[q] = i + (int64_t)q * kJoinBlock < cur.p1;
                        k[q] = ok[q] ? cur.pkeys[i + (int64_t)q * kJoinBlock] : 0u;
                    }
                    local += jn_matches(table, keys, k, ok);
                }
            } else if (!chunks) {
                #pragma unroll
                for (int q = 0; q < kJnPre; ++q)
                    if (threadIdx.x + (int64_t)q * kJoinBlock < pn) local += jn_lookup(table, pk[q], fb);
                for (int64_t i = cur.p0 + kJnPre * kJoinBlock + threadIdx.x; i < cur.p1; i += kJoinBlock)
                    local += jn_lookup(table, cur.pkeys[i], fb);
            }
        }
        if (nb < B) jn_load(nxt.pkeys, nxt.p0, nxt.p1, pk);
        if (chunks) {
            for (int64_t c0 = cur.b0; c0 < cur.b1; c0 += kJoinChunk) {
                const int64_t c1 = std::min<int64_t>(c0 + kJoinChunk, cur.b1);
                __syncthreads();
                for (int i = threadIdx.x; i < kJoinSlots; i += kJoinBlock) table64[i] = 0ull;
                __syncthreads();
                for (int64_t i = c0 + threadIdx.x; i < c1; i += kJoinBlock) join_insert(table64, cur.bkeys[i], 0);
                __syncthreads();
                for (int64_t i = cur.p0 + threadIdx.x; i < cur.p1; i += kJoinBlock)
                    local += join_lookup(table64, cur.pkeys[i], 0);
            }
        }
        cur = nxt;
    }
    join_add_up(local, table64, d_count);
}

}  // namespace

namespace {

// Both relations partitioned into 2^pbits windows by the mix's top bits, then
// joined.  `wide`: 32-bit slots.
int run_one_pass(edpp_ctx* c, const uint32_t* rk, int64_t rn, const uint32_t* sk, int64_t sn, int pbits, bool wide,
                 unsigned long long* d_count) {
    const int W = 1 << pbits;
    JnRel rel[2] = {};
    size_t at = 0;
    auto take = [&at](size_t bytes) {
        const size_t p = at;
        at += (bytes + 255) & ~(size_t)255;
        return p;
    };
    size_t o[2][6];
    for (int i = 0; i < 2; ++i) {
        StGeom& g = rel[i].g;
        rel[i].keys = i ? sk : rk;
        g.n = i ? sn : rn;
        g.shift = 32 - pbits;
        g.W = g.WP = W;
        g.chunks = ceil_div(g.n, (int64_t)kStChunk);
        g.tiles = ceil_div(g.n, (int64_t)kJnTile);
        g.group = st_group(std::max(ceil_div(rn, (int64_t)kJnTile), ceil_div(sn, (int64_t)kJnTile)));
        g.groups = ceil_div(g.tiles, (int64_t)g.group);
        g.xcds = c->xcds;
        o[i][0] = take((size_t)g.n * 4);
        o[i][1] = take((size_t)g.chunks * W * 2);
        o[i][2] = take((size_t)g.tiles * W * 4);
        o[i][3] = take((size_t)g.groups * W * 4);
        o[i][4] = take(((size_t)W + 1) * 4);
        o[i][5] = take((size_t)W * 4);
    }
    void* w;
    int rc = ws_outer_reserve(c, at, &w);
    if (rc) return rc;
    char* p = static_cast<char*>(w);
    for (int i = 0; i < 2; ++i) {
        StGeom& g = rel[i].g;
        rel[i].part = reinterpret_cast<uint32_t*>(p + o[i][0]);
        g.count = reinterpret_cast<uint16_t*>(p + o[i][1]);
        g.rows = reinterpret_cast<uint32_t*>(p + o[i][2]);
        g.gsum = reinterpret_cast<uint32_t*>(p + o[i][3]);
        g.base = reinterpret_cast<uint32_t*>(p + o[i][4]);
        g.total = reinterpret_cast<uint32_t*>(p + o[i][5]);
    }
    const StGeom &g0 = rel[0].g, &g1 = rel[1].g;
    auto both = [](int64_t a, int64_t b) { return dim3((unsigned)std::max(a, b), 2); };
    hipLaunchKernelGGL(k_jn_hist, both(g0.chunks, g1.chunks), dim3(256), 0, c->stream, rel[0], rel[1], d_count);
    launch_st_prefix<kJnCh>(c->stream, g0, &g1);
    EDPP_HIP(c, hipFuncSetAttribute((const void*)k_jn_split, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kJnSplitLds));
    hipLaunchKernelGGL(k_jn_split, both(g0.tiles, g1.tiles), dim3(kStBlock), kJnSplitLds, c->stream, rel[0], rel[1]);
    const size_t lds = wide ? kJnLds : (size_t)kJoinSlots * 8;
    const unsigned grid = (unsigned)std::max(1, std::min(W, std::max(c->cus, 1)));
    const int32_t *rs = reinterpret_cast<const int32_t*>(g0.base), *ss = reinterpret_cast<const int32_t*>(g1.base);
    const auto probe = wide ? k_jn_probe : k_join_probe;
    EDPP_HIP(c, hipFuncSetAttribute((const void*)probe, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    // the partition is the mix's top bits: k_join_probe finds its slots in the low ones
    hipLaunchKernelGGL(probe, dim3(grid), dim3(kJoinBlock), lds, c->stream, rel[0].part, rn, rs, rel[1].part, sn, ss, W,
                       wide ? pbits : 0, d_count);
    EDPP_HIP(c, hipGetLastError());
    return EDPP_OK;
}

}  // namespace

int launch_join_count(edpp_ctx* c, const uint32_t* rk, int64_t rn, const uint32_t* sk, int64_t sn,
                      unsigned long long* d_count) {
    const int64_t small = std::min(rn, sn), large = std::max(rn, sn);
    // One pass: 32-bit slots need 8 partition bits or more for their counts, and
    // from 2^22 keys on 16,384 build keys per partition ask for that many; with
    // fewer keys 64-bit slots and 4096 build keys per partition.  Byte offsets
    // of 31 bits and whole vectors.
    if (small > 0 && small <= (1ll << (kJnMaxBits + 14)) && large < (1ll << 29) && aligned16(rk) && aligned16(sk)) {
        const bool wide = small >= (1ll << 22);
        int bits = wide ? 8 : 1;
        while (bits < kJnMaxBits && (small >> bits) > (wide ? 16384 : kJoinTargetBuild)) ++bits;
        return run_one_pass(c, rk, rn, sk, sn, bits, wide, d_count);
    }
    hipLaunchKernelGGL(k_join_zero, dim3(1), dim3(64), 0, c->stream, d_count);
    EDPP_HIP(c, hipGetLastError());
    if (small == 0) return EDPP_OK;
    // partition bits: about kJoinTargetBuild keys of the smaller side per partition
    int pbits = 0;
    while (pbits < kJoinMaxBits && (small >> pbits) > kJoinTargetBuild) ++pbits;
    const int B = 1 << pbits;
    const size_t rb = ((size_t)rn * 4 + 255) & ~(size_t)255, sb = ((size_t)sn * 4 + 255) & ~(size_t)255;
    const size_t stb = ((size_t)B * 4 + 255) & ~(size_t)255;
    void* w;
    int rc = ws_outer_reserve(c, rb + sb + 2 * stb, &w);
    if (rc) return rc;
    char* base = static_cast<char*>(w);
    uint32_t* rpart = reinterpret_cast<uint32_t*>(base);
    uint32_t* spart = reinterpret_cast<uint32_t*>(base + rb);
    int32_t* rst = reinterpret_cast<int32_t*>(base + rb + sb);
    int32_t* sst = reinterpret_cast<int32_t*>(base + rb + sb + stb);
    // the partitioned relations hold the mixed keys
    rc = launch_split<MixOnLoad>(c, reinterpret_cast<const MixOnLoad*>(rk), reinterpret_cast<MixOnLoad*>(rpart),
                                 nullptr, nullptr, rst, rn, B, EDPP_SPLIT_AUTO);
    if (!rc)
        rc = launch_split<MixOnLoad>(c, reinterpret_cast<const MixOnLoad*>(sk), reinterpret_cast<MixOnLoad*>(spart),
                                     nullptr, nullptr, sst, sn, B, EDPP_SPLIT_AUTO);
    if (rc) return rc;
    const size_t lds = (size_t)kJoinSlots * 8;
    EDPP_HIP(c, hipFuncSetAttribute((const void*)k_join_probe, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    // one persistent workgroup per CU (its table holds the CU's LDS)
    const unsigned grid = (unsigned)std::max(1, std::min(B, std::max(c->cus, 1)));
    hipLaunchKernelGGL(k_join_probe, dim3(grid), dim3(kJoinBlock), lds, c->stream, rpart, rn, rst, spart, sn, sst, B,
                       pbits, d_count);
    EDPP_HIP(c, hipGetLastError());
    return EDPP_OK;
}

}  // namespace edpp
