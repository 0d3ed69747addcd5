// knn_wide_collect.hip -- collect + select kNN of fp32 rows on the fp16 matrix
// cores over rows split in two: bucketed passes over rows longer than 256
// floats, and exact kNN of many queries over rows of up to 128 or more than
// 256
// (src/bucket.cu:4101-4265 top-M semantics: self excluded, (-1, +inf)
// padding, ties by id).
//
// The split.  Row x is scaled by a power of two of its own, 2^k with
// max |x_i| 2^k in [2^14, 2^15), and every element written as h + m: h the
// fp16 nearest to it, m the fp16 nearest to the rest.  h keeps 11 bits and a
// sign, m the next 11, so h + m is the fp32 element to within half of its
// last bit (2^-24 of the element; where m is subnormal, flushed or not,
// within 2^-29 of the row's largest).  A dot product is the sum of h h, h m and m h
// products, each exact in the fp32 accumulator (v_mfma_f32_32x32x16_f16);
// the m m products left out are at most 2^-24 of their terms.  Both are
// below the roundings of an fp32 sum over D terms: measured against 64 bits on
// D 288..1024 (tests/test_gpu_wide_split.py) the distances are as close as
// those of the fp32 kernel (knn_wide_kernel; 1.59 and 1.60 ulps rms at D 960),
// and closer than knn_fused_kernel's (1.9 and 3.1 at D 128).  Integer-valued rows below 2^11
// have m = 0 and give exact sums.
// A row with an element that is not finite has a norm that is not finite
// either: its L2 keys are +inf or NaN, which no list takes, whatever its dot
// products (the inner product of such rows stays on the fp32 kernel).
//
// Three fp16 products cost 3/16 of one fp32 product of the fp32 matrix cores,
// and h and m take the fp32 row's bytes, so moving rows is what there is to
// save: a block is 8 waves with 256 queries (32 per wave, read from L2 chunk
// by chunk) against 192 or 256 pool rows at a time (32-dimension chunks
// double-buffered in LDS, shared by the waves; 6 or 8 accumulator tiles of
// 32 x 32 per wave).  Launches with fewer blocks than the chip has CUs take 4
// waves and 128 queries.  What bounds it (D 960, 2.1e9 pairs, keys not
// collected, variants timed with parts left out): 13.3 ms, without the query
// loads 11.2, without the pool loads 12.1, without either and the barrier 9.2,
// the MFMAs alone 4.9: the LDS reads (every wave reads every pool row), then
// the loads' latency.  Stages of two chunks, half the barriers, were no faster.
// Measured (bucketed pass over 100,003 x 960, 25 buckets, one probe, M 96):
// 20.3 ms on the fp32 kernel, 8.3 here; a 10^6 x 960 build 237 -> 128 ms; exact
// 100-NN of 10,000 queries in 1,000,003 x 100: 40.2 -> 14.1 ms.
//
// Keys at or below a query's threshold go to its candidate slots in HBM as in
// knn_collect.hip.  An unseeded pass first bounds each query's M-th smallest
// key by bisection over the 256 keys of the first pool tile, which the lane
// pair holds in registers.
#include "collect_device.hpp"

#include <algorithm>

namespace gtann {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
constexpr int kMaxSplits = 128;   // pool slices of an exact kNN launch

typedef _Float16 halfx4 __attribute__((ext_vector_type(4)));

constexpr int kSplitChunk = 32;                   // dimensions per chunk: 32 h, then 32 m

// Pool rows per tile.  Rows of up to 256 dimensions sum all chunks in one
// accumulator (their error is below the fp32 kernel's as it is); longer ones
// sum each chunk on its own, which takes the registers of a quarter of the
// tile (D 960, error against 64 bits: 4.8 ulps rms in one accumulator, 1.6 by
// chunks, 1.6 the fp32 kernel).
template <bool PARTS>
struct SplitTile {
    static constexpr int ROWS = PARTS ? 192 : 256;
    static constexpr int TILES = ROWS / kPoolTile;
};
constexpr int kSplitStride = 2 * kSplitChunk + 8; // halves per LDS row: 16 rows' same pieces fill the banks once

// Where the split copy holds chunk c of the row at position p of the member
// list: groups of 32 positions, chunk-major, so that a tile's chunk is a few
// whole 4 KiB pieces (by row id, a 128-byte piece of a row in 512 places per
// chunk, the launch took 2.1 times as long).
__device__ __forceinline__ int64_t split_at(int64_t p, int c, int nch)
{
    return (((p >> 5) * nch + c) * 32 + (p & 31)) * 2 * kSplitChunk;
}

// The rows X[members[p]] (stride Dp; members null: X[p]) to Xs at their positions p: per row and
// chunk 32 h, then 32 m; inv[p] = 2^-k.  *bad counts rows whose |x|^2 is not
// finite.  One wave per position.
__global__ void __launch_bounds__(256) split_rows_kernel(const float* __restrict__ X, const float* __restrict__ nrm,
                                                         const int32_t* __restrict__ members, int64_t N, int Dp,
                                                         _Float16* __restrict__ Xs, float* __restrict__ inv,
                                                         unsigned int* __restrict__ bad)
{
    const int lane = threadIdx.x & 63;
    const int64_t pos = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (pos >= N) return;
    const int64_t row = members ? members[pos] : pos;
    const float4* x = reinterpret_cast<const float4*>(X + row * Dp);
    const int n4 = Dp >> 2;
    float4 v[4];                                   // Dp <= 1024: four float4 per lane
    float mx = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        v[t] = lane + 64 * t < n4 ? x[lane + 64 * t] : make_float4(0.f, 0.f, 0.f, 0.f);
        mx = fmaxf(fmaxf(fmaxf(mx, fabsf(v[t].x)), fmaxf(fabsf(v[t].y), fabsf(v[t].z))), fabsf(v[t].w));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    int e = 0;
    const bool finite = mx < INFINITY;
    if (finite && mx > 0.f) frexpf(mx, &e);        // mx < 2^e
    // (at most 2^126: the scale back stays a normal float; every float element
    // is then a multiple of 2^-23, which the two parts hold as well)
    const int k = finite && mx > 0.f ? min(15 - e, 126) : 0;
    auto scaled = [&](float y) -> float { return finite ? ldexpf(y, k) : 0.f; };
    const int nch = Dp / kSplitChunk;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int q = lane + 64 * t;
        if (q < n4) {
            const float y[4] = {scaled(v[t].x), scaled(v[t].y), scaled(v[t].z), scaled(v[t].w)};
            halfx4 h, m;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                h[i] = static_cast<_Float16>(y[i]);
                m[i] = static_cast<_Float16>(y[i] - static_cast<float>(h[i]));
            }
            const int d = 4 * q;                   // dims d .. d + 3 of chunk d / 32
            _Float16* c = Xs + split_at(pos, d / kSplitChunk, nch) + d % kSplitChunk;
            *reinterpret_cast<halfx4*>(c) = h;
            *reinterpret_cast<halfx4*>(c + kSplitChunk) = m;
        }
    }
    if (lane == 0) {
        inv[pos] = ldexpf(1.f, -k);
        if (!(nrm[row] < INFINITY)) atomicAdd(bad, 1u);
    }
}

__global__ void split_clear_kernel(unsigned int* bad) { *bad = 0u; }

void launch_split_rows(const float* X, const float* nrm, const int32_t* members, int64_t N, int Dp, uint16_t* Xs,
                       float* inv, unsigned int* bad, hipStream_t s)
{
    GT_REQUIRE(Dp % kSplitChunk == 0 && Dp <= 1024, "split rows: padded dimension");
    hipLaunchKernelGGL(split_clear_kernel, dim3(1), dim3(1), 0, s, bad);
    if (N > 0)
        hipLaunchKernelGGL(split_rows_kernel, dim3(static_cast<unsigned>(ceil_div(N, int64_t(4)))), dim3(256), 0, s, X,
                           nrm, members, N, Dp, reinterpret_cast<_Float16*>(Xs), inv, bad);
    GT_HIP(hipGetLastError());
}

__global__ void __launch_bounds__(256) iota_kernel(int32_t* p, int64_t n)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) p[i] = static_cast<int32_t>(i);
}

void launch_iota(int32_t* p, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(iota_kernel, dim3(static_cast<unsigned>(ceil_div(n, int64_t(256)))), dim3(256), 0, s, p, n);
    GT_HIP(hipGetLastError());
}

template <int NW, bool PARTS>
struct WideCollectSmem {
    static constexpr int kSplitRows = SplitTile<PARTS>::ROWS;
    _Float16 tile[2][kSplitRows][kSplitStride];
    float tnorm[2][kSplitRows];     // |p|^2 (L2) or 0 (IP); +inf past the slice end
    float tinv[2][kSplitRows];      // 2^-k of the row
    int32_t trow[2][kSplitRows];    // pool row id, -1 past the slice end
    CollectWave wv[NW];
};

template <int METRIC, int NW, bool PARTS>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 8 ? 2 : 1)))
knn_wide_collect_kernel(KnnArgs a, const _Float16* __restrict__ Xs, const float* __restrict__ inv,
                        const int32_t* __restrict__ p_pos, int q_by_row)
{
    extern __shared__ __align__(16) unsigned char smem[];
    using Smem = WideCollectSmem<NW, PARTS>;
    Smem& sm = *reinterpret_cast<Smem*>(smem);
    constexpr int kSplitRows = SplitTile<PARTS>::ROWS, kSplitTiles = SplitTile<PARTS>::TILES;
    constexpr int T = 64 * NW;
    constexpr int PT = kSplitRows * 8 / T;          // 16-byte pieces of a chunk's rows per thread
    static_assert(PT * T == kSplitRows * 8, "whole pieces");
    constexpr int RS = T / 8;                       // rows between a thread's pieces

    const int per = a.n_items / 8;
    const int item_idx = static_cast<int>(blockIdx.x % 8) * per + static_cast<int>(blockIdx.x / 8);
    if (item_idx >= a.n_items) return;
    const WorkItem it = a.items[item_idx];
    if (it.q_count <= 0) return;

    const int Dp = a.Dp;
    const int nch = Dp / kSplitChunk;
    const int tid = threadIdx.x;
    const int w = tid >> 6, lane = tid & 63, j = lane & 31, h = lane >> 5;
    const int qlocal = w * kQueriesPerWave + j;
    const bool qvalid = qlocal < it.q_count;
    const int64_t qi = it.q_begin + qlocal;
    const int32_t qrow = qvalid ? (a.q_rows ? a.q_rows[qi] : static_cast<int32_t>(qi)) : 0;
    const float qn = (qvalid && METRIC == 0) ? a.nq[qrow] : 0.f;
    const int64_t qpos = q_by_row ? qrow : qvalid ? qi : it.q_begin;
    const float qinv = inv[qpos];

    CollectState st;
    float seed = FLT_MAX;
    // the seed is read from the output row (the query row unless the item has an out_base)
    const int64_t orow = it.out_base >= 0 ? it.out_base + qlocal : static_cast<int64_t>(qrow);
    if (qvalid && a.seed_d) seed = fminf(a.seed_d[orow * a.seed_ld + a.seed_ld - 1], FLT_MAX);
    st.thr = qvalid ? seed : -INFINITY;
    st.thr_id = 0xffffffffu;
    st.cnt = 0;
    st.self = a.exclude_self ? qrow : -2;
    st.orow = orow;
    CollectWave& W = sm.wv[w];
    publish_state(W, lane, qvalid, qn, st);

    const int pcount = it.p_count;
    const int nst = (pcount + kSplitRows - 1) / kSplitRows;
    // the pool-list entry scanned at p (< pcount)
    auto pool_at = [&](int p) -> int64_t {
        p += it.p_rot;
        if (p >= pcount) p -= pcount;
        return it.p_begin + p;
    };

    // thread tid stages 16-byte piece tid % 8 of rows tid / 8 + RS u (rows past
    // the slice hold the last row's values: their norm is +inf and their id -1)
    const int piece = tid & 7, r0 = tid >> 3;
    int32_t rid[PT], rid_n[PT];   // their positions in the member list
    uint4 pre[PT];
    auto set_ids = [&](int stile, int32_t (&ids)[PT]) {
#pragma unroll
        for (int u = 0; u < PT; ++u) {
            const int64_t pl = pool_at(min(stile * kSplitRows + r0 + RS * u, pcount - 1));
            ids[u] = p_pos ? p_pos[pl] : static_cast<int32_t>(pl);
        }
    };
    auto load_pool = [&](bool next, int c) {
#pragma unroll
        for (int u = 0; u < PT; ++u) {
            const int32_t p = next ? rid_n[u] : rid[u];
            const uint4 v = *reinterpret_cast<const uint4*>(Xs + split_at(p, c, nch) + 8 * piece);
            pre[u] = make_uint4(v.x, v.y, v.z, v.w);
        }
    };
    auto store_pool = [&](int buf) {
#pragma unroll
        for (int u = 0; u < PT; ++u) *reinterpret_cast<uint4*>(&sm.tile[buf][r0 + RS * u][8 * piece]) = pre[u];
    };
    // the query's chunk: h of dims 8h.., 16 + 8h.., then m
    halfx8 qc[4], qx[4];
    auto load_q = [&](int c, halfx8 (&dst)[4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s) dst[s] = *reinterpret_cast<const halfx8*>(Xs + split_at(qpos, c, nch) + 8 * h + 16 * s);
    };
    // ids, norms and scales of tile stile's row tid
    auto tile_meta = [&](int stile, int32_t& id, float& n, float& iv) {
        id = -1;
        n = INFINITY;
        iv = 1.f;
        const int p = stile * kSplitRows + tid;
        if (tid < kSplitRows && p < pcount) {
            const int64_t pl = pool_at(p);
            id = a.p_rows ? a.p_rows[pl] : static_cast<int32_t>(pl);
            n = METRIC == 0 ? a.np[id] : 0.f;
            iv = inv[p_pos ? p_pos[pl] : pl];
        }
    };
    static_assert(T >= kSplitRows || T == 256, "one row's ids per thread");

    if (nst > 0) {
        set_ids(0, rid);
        set_ids(1, rid_n);
        int32_t nrow;
        float nnrm, ninv;
        tile_meta(0, nrow, nnrm, ninv);
        if (tid < kSplitRows) {
            sm.trow[0][tid] = nrow;
            sm.tnorm[0][tid] = nnrm;
            sm.tinv[0][tid] = ninv;
        }
        load_pool(false, 0);
        store_pool(0);
        load_q(0, qc);
        __syncthreads();
    }

    int g = 0;
    for (int stile = 0; stile < nst; ++stile) {
        floatx16 acc[kSplitTiles];
#pragma unroll
        for (int u = 0; u < kSplitTiles; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[u][r] = 0.f;
        int32_t nrow;
        float nnrm, ninv;
        tile_meta(stile + 1, nrow, nnrm, ninv);
#pragma unroll 1
        for (int c = 0; c < nch; ++c) {
            const int buf = g & 1;
            const bool last = c + 1 == nch;
            load_pool(last, last ? 0 : c + 1);
            load_q(last ? 0 : c + 1, qx);
            // the next chunk's loads stay ahead of this chunk's MFMAs
            __builtin_amdgcn_sched_barrier(0);
            // A = pool row u*32 + (lane%32), B = query lane%32, the small
            // products first; PARTS: the chunk's sum is added to the running
            // dot, so that the rounding error grows with sqrt(chunks)
#pragma unroll
            for (int u = 0; u < kSplitTiles; ++u) {
                halfx8 av[4];
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    av[s] = *reinterpret_cast<const halfx8*>(&sm.tile[buf][kPoolTile * u + j][8 * h + 16 * s]);
                floatx16 part;
#pragma unroll
                for (int r = 0; r < 16; ++r) part[r] = PARTS ? 0.f : acc[u][r];
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[2], qc[0], part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[3], qc[1], part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[0], qc[2], part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[1], qc[3], part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[0], qc[0], part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[1], qc[1], part, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[u][r] = PARTS ? acc[u][r] + part[r] : part[r];
            }
            store_pool(buf ^ 1);
            __syncthreads();
#pragma unroll
            for (int s = 0; s < 4; ++s) qc[s] = qx[s];
            ++g;
        }
        if (tid < kSplitRows) {
            sm.trow[(stile + 1) & 1][tid] = nrow;
            sm.tnorm[(stile + 1) & 1][tid] = nnrm;
            sm.tinv[(stile + 1) & 1][tid] = ninv;
        }
#pragma unroll
        for (int u = 0; u < PT; ++u) rid[u] = rid_n[u];
        set_ids(stile + 2, rid_n);

        // the keys, in place: lane (j, h) holds rows 8g + 4h + e of every tile
        const int sb = stile & 1;
#pragma unroll
        for (int u = 0; u < kSplitTiles; ++u)
#pragma unroll
            for (int gg = 0; gg < 4; ++gg) {
                const float4 pn = *reinterpret_cast<const float4*>(&sm.tnorm[sb][kPoolTile * u + 8 * gg + 4 * h]);
                const float4 pi = *reinterpret_cast<const float4*>(&sm.tinv[sb][kPoolTile * u + 8 * gg + 4 * h]);
                const float n4[4] = {pn.x, pn.y, pn.z, pn.w}, i4[4] = {pi.x, pi.y, pi.z, pi.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // powers of two: exact (their product alone may underflow where the dot does not)
                    const float dot = (acc[u][4 * gg + e] * qinv) * i4[e];
                    acc[u][4 * gg + e] = METRIC == 0 ? fmaf(-2.f, dot, n4[e] + qn) : fmaf(-1.f, dot, n4[e]);
                }
            }
        if (stile == 0 && !a.seed_d) {
            // a bound on the M-th smallest key: bisection between the
            // smallest and the largest of the pair's 256 keys (the query
            // itself among them: one more than M keys at or below it)
            float lo = INFINITY, hi = -INFINITY;
            int n = 0;
#pragma unroll
            for (int u = 0; u < kSplitTiles; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float k = acc[u][r];
                    const bool in = k < INFINITY && k > -INFINITY;
                    lo = in ? fminf(lo, k) : lo;
                    hi = in ? fmaxf(hi, k) : hi;
                    n += in ? 1 : 0;
                }
            lo = fminf(lo, __shfl_xor(lo, 32));
            hi = fmaxf(hi, __shfl_xor(hi, 32));
            n += __shfl_xor(n, 32);
            const bool enough = n > a.M;
            for (int i = 0; i < 12; ++i) {
                const float mid = 0.5f * lo + 0.5f * hi;
                int c = 0;
#pragma unroll
                for (int u = 0; u < kSplitTiles; ++u)
#pragma unroll
                    for (int r = 0; r < 16; ++r) c += acc[u][r] <= mid ? 1 : 0;
                c += __shfl_xor(c, 32);
                if (c > a.M) hi = mid;
                else lo = mid;
            }
            if (qvalid && enough && hi < st.thr) st.thr = hi;
            publish_state(W, lane, qvalid, qn, st);
        }
#pragma unroll
        for (int u = 0; u < kSplitTiles; ++u) {
            float d[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) d[r] = acc[u][r];
            collect_keys_f32(a, W, d, &sm.trow[sb][kPoolTile * u], lane, qvalid, qn, st);
        }
    }
    if (qvalid && h == 0) a.cand_cnt[st.orow] = st.cnt;
    if (a.stats && qvalid && h == 0) atomicAdd(a.stats, static_cast<unsigned long long>(st.cnt));
}

// ------------------------------------------------------------ selection, long lists

// Sorts the wave's 64 KPL keys ascending, element KPL lane + r in k[r]
// (bitonic; partners of other lanes through shuffles).
template <int KPL>
__device__ __forceinline__ void wave_sort(uint64_t (&k)[KPL], int lane)
{
    constexpr int N = 64 * KPL;
#pragma unroll
    for (int size = 2; size <= N; size <<= 1) {
#pragma unroll
        for (int d = size >> 1; d > 0; d >>= 1) {
            if (d < KPL) {
#pragma unroll
                for (int r = 0; r < KPL; ++r)
                    if ((r & d) == 0) {
                        const bool up = ((KPL * lane + r) & size) == 0;
                        const bool sw = (k[r + d] < k[r]) == up;
                        const uint64_t lo = sw ? k[r + d] : k[r];
                        k[r + d] = sw ? k[r] : k[r + d];
                        k[r] = lo;
                    }
            } else {
                const int ld = d / KPL;
                const bool low = (lane & ld) == 0;
#pragma unroll
                for (int r = 0; r < KPL; ++r) {
                    const bool up = ((KPL * lane + r) & size) == 0;
                    const uint64_t o = shfl_xor_u64(k[r], ld);
                    const bool take = (o < k[r]) == (low == up);   // distinct keys or equal fillers
                    k[r] = take ? o : k[r];
                }
            }
        }
    }
}

// Row's top M (1..128) of its cnt[row] keys, ascending: one wave per row
// sorts them (2 or 4 keys per lane).  Rows of at most skip_le keys are neither
// sorted nor written.
__global__ void __launch_bounds__(256) knn_sort_select_kernel(const uint64_t* __restrict__ cand,
                                                              const int32_t* __restrict__ cnt, int64_t rows, int M,
                                                              int skip_le, int32_t* __restrict__ out_ids,
                                                              float* __restrict__ out_d)
{
    const int lane = threadIdx.x & 63;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int n = __builtin_amdgcn_readfirstlane(min(cnt[row], kCollectCap));
    if (n <= skip_le) return;
    const uint64_t* src = cand + row * kCollectCap;
    auto go = [&](auto kpl) __attribute__((always_inline)) {
        constexpr int KPL = decltype(kpl)::value;
        uint64_t k[KPL];
#pragma unroll
        for (int r = 0; r < KPL; ++r) k[r] = KPL * lane + r < n ? src[KPL * lane + r] : kNoKey;
        if (n > 0) wave_sort(k, lane);
#pragma unroll
        for (int r = 0; r < KPL; ++r) {
            const int p = KPL * lane + r;
            if (p < M) {
                out_ids[row * M + p] = k[r] == kNoKey ? -1 : static_cast<int32_t>(static_cast<uint32_t>(k[r]));
                out_d[row * M + p] = k[r] == kNoKey ? INFINITY : o2f(static_cast<uint32_t>(k[r] >> 32));
            }
        }
    };
    if (n <= 128) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 4>{});
}

void launch_sort_select(const uint64_t* cand, const int32_t* cnt, int64_t rows, int M, int skip_le, int32_t* out_ids,
                        float* out_d, hipStream_t s)
{
    GT_REQUIRE(M >= 1 && M <= 128 && kCollectCap == 256, "sort selection: list length");
    if (rows <= 0) return;
    hipLaunchKernelGGL(knn_sort_select_kernel, dim3(static_cast<unsigned>(ceil_div(rows, int64_t(4)))), dim3(256), 0, s,
                       cand, cnt, rows, M, skip_le, out_ids, out_d);
    GT_HIP(hipGetLastError());
}

// The top M of each query's candidate lists over `splits` pool slices (list s
// of query q: row s nq + q), ascending.  One block per query: the distances'
// ordered bits in LDS, a bound with at least M and at most 256 keys at or below
// it by bisection (by (distance, id) where more than 256 tie), those keys
// sorted by the first wave.
__global__ void __launch_bounds__(256) knn_split_select_kernel(const uint64_t* __restrict__ cand,
                                                               const int32_t* __restrict__ cnt, int64_t nq, int splits,
                                                               int M, int32_t* __restrict__ out_ids,
                                                               float* __restrict__ out_d)
{
    extern __shared__ __align__(16) unsigned char smem[];
    uint32_t* key = reinterpret_cast<uint32_t*>(smem);   // up to splits * kCollectCap
    __shared__ int first[kMaxSplits + 1];
    __shared__ uint64_t pick[kCollectCap];
    __shared__ uint32_t ext[2][4];
    __shared__ int sums[4], npick;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t q = blockIdx.x;
    if (tid < splits) first[tid + 1] = min(cnt[tid * nq + q], kCollectCap);
    if (tid == 0) { first[0] = 0; npick = 0; }
    __syncthreads();
    if (tid == 0)
        for (int s = 0; s < splits; ++s) first[s + 1] += first[s];
    __syncthreads();
    const int total = first[splits];
    uint32_t mx = 0, mn = 0xFFFFFFFFu;
    for (int s = w; s < splits; s += 4) {
        const int n = first[s + 1] - first[s];
        for (int i = lane; i < n; i += 64) {
            const uint32_t d = static_cast<uint32_t>(cand[(s * nq + q) * kCollectCap + i] >> 32);
            key[first[s] + i] = d;
            mx = max(mx, d);
            mn = min(mn, d);
        }
    }
    mx = wave_extreme_u32<true>(mx);
    mn = wave_extreme_u32<false>(mn);
    if (lane == 0) { ext[0][w] = mx; ext[1][w] = mn; }
    __syncthreads();
    uint32_t hi = max(max(ext[0][0], ext[0][1]), max(ext[0][2], ext[0][3]));
    uint32_t lo = min(min(ext[1][0], ext[1][1]), min(ext[1][2], ext[1][3])) - 1u;
    int n = total;
    auto block_sum = [&](int c) -> int {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
        __syncthreads();   // the last sum was read
        if (lane == 0) sums[w] = c;
        __syncthreads();
        return sums[0] + sums[1] + sums[2] + sums[3];
    };
    while (n > kCollectCap && hi - lo > 1u) {   // uniform: every thread holds the same bounds
        const uint32_t mid = lo + ((hi - lo) >> 1);
        int c = 0;
        for (int i = tid; i < total; i += 256) c += key[i] <= mid ? 1 : 0;
        c = block_sum(c);
        if (c < M) lo = mid;
        else { hi = mid; n = c; }
    }
    uint64_t K = (static_cast<uint64_t>(hi) << 32) | 0xFFFFFFFFu;
    if (n > kCollectCap) {
        // ties at distance hi: the ids decide (fewer than M keys lie below hi)
        uint32_t ilo = 0, ihi = 0xFFFFFFFFu;   // at least M keys with (hi, id <= ihi)
        while (ilo < ihi) {
            const uint32_t mid = ilo + ((ihi - ilo) >> 1);
            const uint64_t t = (static_cast<uint64_t>(hi) << 32) | mid;
            int c = 0;
            for (int s = w; s < splits; s += 4)
                for (int i = lane; i < first[s + 1] - first[s]; i += 64) c += cand[(s * nq + q) * kCollectCap + i] <= t ? 1 : 0;
            c = block_sum(c);
            if (c >= M) ihi = mid;
            else ilo = mid + 1;
        }
        K = (static_cast<uint64_t>(hi) << 32) | ihi;
    }
    __syncthreads();
    for (int s = w; s < splits; s += 4)
        for (int i = lane; i < first[s + 1] - first[s]; i += 64) {
            const uint64_t k = cand[(s * nq + q) * kCollectCap + i];
            if (k <= K) pick[atomicAdd(&npick, 1)] = k;
        }
    __syncthreads();
    if (w > 0) return;
    constexpr int KPL = kCollectCap / 64;
    uint64_t k[KPL];
#pragma unroll
    for (int r = 0; r < KPL; ++r) k[r] = KPL * lane + r < npick ? pick[KPL * lane + r] : kNoKey;
    wave_sort(k, lane);
#pragma unroll
    for (int r = 0; r < KPL; ++r) {
        const int p = KPL * lane + r;
        if (p < M) {
            out_ids[q * M + p] = k[r] == kNoKey ? -1 : static_cast<int32_t>(static_cast<uint32_t>(k[r]));
            out_d[q * M + p] = k[r] == kNoKey ? INFINITY : o2f(static_cast<uint32_t>(k[r] >> 32));
        }
    }
}

void launch_split_select(const uint64_t* cand, const int32_t* cnt, int64_t nq, int splits, int M, int32_t* out_ids,
                         float* out_d, hipStream_t s)
{
    GT_REQUIRE(M >= 1 && M <= 128 && splits >= 1 && splits <= kMaxSplits && nq < (int64_t(1) << 31), "split selection");
    if (nq <= 0) return;
    const size_t lds = static_cast<size_t>(splits) * kCollectCap * 4;
    GT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&knn_split_select_kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    hipLaunchKernelGGL(knn_split_select_kernel, dim3(static_cast<unsigned>(nq)), dim3(256), lds, s, cand, cnt, nq, splits,
                       M, out_ids, out_d);
    GT_HIP(hipGetLastError());
}

// Queries per block of a launch over n_queries queries: 256 (8 waves) where
// that gives every CU a block, else 128.
int wide_queries_per_block(int64_t n_queries) { return n_queries >= int64_t(256) * 256 ? 256 : 128; }

// Xs, inv: the split rows by position; p_pos: the position of every pool-list
// entry (null: itself).  Query i's position is i, its place in the member list
// a.q_rows, or with q_by_row its row id (rows split in their own order).
void launch_wide_collect(const KnnArgs& a, int qpb, const uint16_t* Xs, const float* inv, const int32_t* p_pos,
                         bool q_by_row, hipStream_t s)
{
    GT_REQUIRE((p_pos != nullptr) == (a.p_rows != nullptr) && a.n_items % 8 == 0 && a.Dp % kSplitChunk == 0 && a.cand && a.cand_cnt && (qpb == 128 || qpb == 256),
               "wide collect launch");
    if (a.n_items <= 0) return;
    const _Float16* x = reinterpret_cast<const _Float16*>(Xs);
    auto go = [&](auto kernel, int waves, size_t lds) {
        GT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(lds)));
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.n_items)), dim3(static_cast<unsigned>(64 * waves)), lds, s,
                           a, x, inv, p_pos, q_by_row ? 1 : 0);
    };
    auto by_metric = [&](auto nw, auto parts) {
        constexpr int NW = decltype(nw)::value;
        constexpr bool P = decltype(parts)::value;
        if (a.metric == 0) go(&knn_wide_collect_kernel<0, NW, P>, NW, sizeof(WideCollectSmem<NW, P>));
        else go(&knn_wide_collect_kernel<1, NW, P>, NW, sizeof(WideCollectSmem<NW, P>));
    };
    auto by_dim = [&](auto nw) {
        if (a.Dp > 256) by_metric(nw, std::true_type{});
        else by_metric(nw, std::false_type{});
    };
    if (qpb == 256) by_dim(std::integral_constant<int, 8>{});
    else by_dim(std::integral_constant<int, 4>{});
    GT_HIP(hipGetLastError());
}

}  // namespace gtann
