// collect_device.hpp -- device pieces shared by the collect kernels
// (knn_collect.hip: int8 and fp32 rows in LDS tiles; knn_wide_collect.hip:
// rows split into three bf16 parts).
#pragma once

#include "knn_device.hpp"

#include <type_traits>

namespace gtann {

// Per-wave staging of a tile's candidates: every lane's 16 accumulators
// (16-byte chunks swizzled by lane so that a wave's 128-bit stores spread
// over the banks), one 16-bit code (lane << 4 | element) per accumulator at
// or above its lane's pass floor (plus a spare slot per lane), the wave's
// queries' slot counters and the query state the dense pass reads.
constexpr int kCodeSpare = 64 * 16;   // first of the 64 per-lane spare code slots

struct CollectWave {
    int32_t stash[64 * 16];
    uint16_t code[kCodeSpare + 64];
    int32_t qcnt[kQueriesPerWave];
    float4 qst[kQueriesPerWave];          // |q|^2, threshold, threshold id (bits), self (bits)
    int64_t qrow_out[kQueriesPerWave];    // output row
};

__device__ __forceinline__ int stash_index(int lane, int r)
{
    return lane * 16 + (((r >> 2) ^ ((lane >> 1) & 3)) << 2) + (r & 3);
}

// Per-lane view of one query (lanes j and j + 32 hold identical copies).
struct CollectState {
    float thr;          // a key passes iff (d, id) <= (thr, thr_id)
    uint32_t thr_id;    // 0xffffffff: every id at distance thr
    int32_t cnt;        // keys in the query's slots
    int32_t self;       // id that must not be kept (the query itself), -2 if none
    int64_t orow;       // output row
};

__device__ __forceinline__ bool key_passes(float d, int32_t id, const CollectState& st)
{
    return d < st.thr || (d == st.thr && static_cast<uint32_t>(id) <= st.thr_id);
}

// Drops the largest of query q's cnt (> M) keys: its slots keep the M smallest
// and at most kCompactSlack more (up to kCollectCap - 64 in all where more tie
// at the last distance), and the largest distance kept becomes its threshold.  The distance is found by bisection over the ordered bits of the
// keys' distances (about 7 steps of a compare and a bit count per 64 keys; the
// exact M-th key takes 64 such steps over both words, 1,100 instructions, and
// made up most of the wide kernel's vector work).  Only where more keys tie
// there than the slots can spare is it the M-th key in (distance, id) order.
// Called by all 64 lanes; q is uniform.
constexpr int kCompactSlack = 16;

__device__ __forceinline__ void collect_compact(const KnnArgs& a, int lane, int q, CollectState& st)
{
    const int cntq = __builtin_amdgcn_readlane(st.cnt, q);
    const int64_t orow = static_cast<int64_t>(
        (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(st.orow >> 32), q))) << 32) |
        static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(st.orow), q)));
    uint64_t* slots = a.cand + orow * kCollectCap;
    // the slots were stored by lanes q and q + 32: complete, then visible to
    // the wave (workgroup-scope loads)
    wait_vmem();
    wave_sync();
    constexpr int KPL = kCollectCap / 64;   // slots per lane
    static_assert(kCollectCap % 64 == 0, "whole slots per lane");
    uint64_t k[KPL];
    uint32_t dmax = 0, dmin = 0xFFFFFFFFu;
#pragma unroll
    for (int i = 0; i < KPL; ++i) {
        const bool in = lane + 64 * i < cntq;
        k[i] = in ? __hip_atomic_load(slots + lane + 64 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : kNoKey;
        const uint32_t d = static_cast<uint32_t>(k[i] >> 32);
        dmax = in ? max(dmax, d) : dmax;
        dmin = in ? min(dmin, d) : dmin;
    }
    const int M = a.M;
    // fewer than M keys at distances up to lo, at least M (n) up to hi; no
    // real distance has the bits 0
    uint32_t hi = wave_extreme_u32<true>(dmax), lo = wave_extreme_u32<false>(dmin) - 1u;
    int n = cntq;
    while (hi - lo > 1u && n > M + kCompactSlack) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        int c = 0;
#pragma unroll
        for (int i = 0; i < KPL; ++i) c += __popcll(__ballot(static_cast<uint32_t>(k[i] >> 32) <= mid));
        if (c < M) {
            lo = mid;
        } else {
            hi = mid;
            n = c;
        }
    }
    uint64_t K = (static_cast<uint64_t>(hi) << 32) | 0xFFFFFFFFu;
    if (n > kCollectCap - 4 * 16) {
        // ties: the M-th smallest key, the largest K with fewer than M keys below it
        K = 0;
        for (int b = 63; b >= 0; --b) {
            const uint64_t t = K | (1ull << b);
            int below = 0;
#pragma unroll
            for (int i = 0; i < KPL; ++i) below += __popcll(__ballot(k[i] < t));
            if (below < M) K = t;
        }
        n = M;
    }
    const uint64_t lt = (1ull << lane) - 1ull;
    int base = 0;
#pragma unroll
    for (int i = 0; i < KPL; ++i) {
        const bool p = k[i] <= K && k[i] != kNoKey;
        const uint64_t m = __ballot(p);
        if (p) slots[base + __popcll(m & lt)] = k[i];
        base += __popcll(m);
    }
    if ((lane & 31) == q) {
        st.cnt = n;
        st.thr = o2f(static_cast<uint32_t>(K >> 32));
        st.thr_id = static_cast<uint32_t>(K);
    }
    if (a.stats && lane == 0) atomicAdd(a.stats + 1, 1ull);
}

// The query state the dense pass reads, published by lanes 0..31.
__device__ __forceinline__ void publish_state(CollectWave& W, int lane, bool qvalid, float qn, const CollectState& st)
{
    if (lane < kQueriesPerWave) {
        W.qst[lane] = make_float4(qn, qvalid ? st.thr : -INFINITY, __uint_as_float(st.thr_id), __int_as_float(st.self));
        W.qrow_out[lane] = st.orow;
    }
}

// One finished 32x32 tile whose lane (j, h) holds the fp32 keys of query j
// against the tile's rows 8g + 4h + e in d[4g + e]: a code is written for
// every key at or below the query's threshold (the stash holds the keys
// themselves), and the exact (key, id) test and the append are made per code.
__device__ __forceinline__ void collect_keys_f32(const KnnArgs& a, CollectWave& W, const float (&d)[16],
                                                 const int32_t* tr, int lane, bool qvalid, float qn, CollectState& st)
{
    float dmin = d[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) dmin = fminf(dmin, d[r]);
    if (!__ballot(dmin <= st.thr)) return;
    uint64_t need = __ballot(qvalid && st.cnt > kCollectCap - 2 * 16) & 0xffffffffull;
    if (need) {
        while (need) {
            const int q = __ffsll(static_cast<unsigned long long>(need)) - 1;
            need &= need - 1;
            collect_compact(a, lane, q, st);
        }
        publish_state(W, lane, qvalid, qn, st);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        *reinterpret_cast<int4*>(&W.stash[stash_index(lane, 4 * c)]) =
            make_int4(__float_as_int(d[4 * c]), __float_as_int(d[4 * c + 1]), __float_as_int(d[4 * c + 2]),
                      __float_as_int(d[4 * c + 3]));
    if (lane < kQueriesPerWave) W.qcnt[lane] = st.cnt;
    int c = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) c += d[r] <= st.thr ? 1 : 0;
    const int incl = wave_incl_scan(c);
    const int total = __builtin_amdgcn_readlane(incl, 63);
    int pos = incl - c;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const bool p = d[r] <= st.thr;
        W.code[p ? pos : kCodeSpare + lane] = static_cast<uint16_t>((lane << 4) | r);
        pos += p ? 1 : 0;
    }
    wave_sync();
    for (int k = lane; k - lane < total; k += 64) {
        if (k < total) {
            const int code = W.code[k];
            const int src = code >> 4, r = code & 15;
            const float dk = __int_as_float(W.stash[stash_index(src, r)]);
            const int q = src & 31;
            const int row = 8 * (r >> 2) + 4 * (src >> 5) + (r & 3);
            const int32_t id = tr[row];
            const float4 Q = W.qst[q];
            const bool ok = id >= 0 && id != __float_as_int(Q.w) &&
                            (dk < Q.y || (dk == Q.y && static_cast<uint32_t>(id) <= __float_as_uint(Q.z)));
            if (ok) {
                const int slot = atomicAdd(&W.qcnt[q], 1);
                a.cand[W.qrow_out[q] * kCollectCap + slot] = pack_key(dk, id);
            }
        }
    }
    wave_sync();
    st.cnt = W.qcnt[lane & 31];
}

}  // namespace gtann
