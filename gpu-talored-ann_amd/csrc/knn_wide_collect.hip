// knn_wide_collect.hip -- collect + select kNN of fp32 rows on the bf16 matrix
// cores over rows split in three: bucketed passes over rows longer than 256
// floats, and exact kNN of many queries over rows of up to 128 or more than
// 256
// (src/bucket.cu:4101-4265 top-M semantics: self excluded, (-1, +inf)
// padding, ties by id).
//
// The split.  Row x is scaled by a power of two of its own, 2^k with
// |x| 2^k in [2^56, 2^57), and every element written as h + m + l: h the bf16
// nearest to it, m the bf16 nearest to the rest, l what is left.  Each takes
// the next 8 of the element's 24 bits, so the three are the element exactly
// (while it is above 2^-110 of |x|: l is then a normal number).  A dot product
// is the sum of the products h h, h m, m h, h l, l h and m m, each exact in
// the fp32 accumulator (v_mfma_f32_32x32x16_bf16); the three left out are at
// most 2^-26 of their terms, a quarter of a product's own rounding in fp32.
// So nothing is lost whatever the rows hold: few dimensions, few non-zeros,
// whole numbers (products below 2^24 have no part in those left out: one
// factor is below 2^12 and then has no l, and has no m where the other has an
// l).  Two fp16 parts and three products, half the matrix work, lose the
// element's last bit and m m: a row of one element 3001 then lay at distance 2
// from its own duplicate, and rows of 1 to 4 elements had twice the fp32
// kernel's error.  Measured against 64 bits (tests/test_gpu_wide_split.py,
// tests/test_gpu_knn_exact_split.py): never above the fp32 kernels' error.
// The inner product asks for every term's own bits: there a row with a
// non-zero element below 2^-105 of |x| (a product of two could leave a part
// below the normal numbers), or a norm that is not finite, sends the launch to
// the fp32 kernel.  L2 keys add |q|^2 + |p|^2, whose rounding is far above.
// A row with an element that is not finite has a norm that is not finite
// either: its L2 keys are +inf or NaN, which no list takes, whatever its dot
// products.
//
// Six bf16 products cost 6/16 of one fp32 product of the fp32 matrix cores.
// Rows move as scaled floats, in an order of their own (piece_at), and are
// split on their way into LDS and into the query operands while the matrix
// cores are busy: a block is 8 waves with 256 queries (32 per wave, read from
// L2 chunk by chunk) against 192 pool rows at a time (32-dimension chunks
// double-buffered in LDS, shared by the waves; 6 accumulator tiles of 32 x 32
// per wave).  Short launches take 4 waves and 128 queries
// (wide_queries_per_block).  A copy of the three parts, 6 bytes per element, was
// slower: bucketed pass below 13.0 ms, build 187.
// What bounds it (a 10^6 x 960 build, counters): six products per element at
// 963 TFLOP/s, 85 % of what a large bf16 product reaches on the card (1.13
// PFLOP/s); the matrix cores are busy 54 % of the time, beside the sums' 32
// additions per tile, the split and the barrier of each chunk.  A pass of some
// 400 blocks, a bucket's on one XCD, holds the CUs only 52 % of the time.
// Measured: bucketed pass over 100,003 x 960 (25 buckets, one probe, M 96)
// 20.8 ms on the fp32 kernel, 12.4 to 15.0 here (by GPU); the build 237 -> 166
// to 172 ms; exact 100-NN of 10,000 queries in 1,000,003 x 100 40.2 -> 19.3 ms.
// (With two fp16 parts, which lose bits: 8.4, 128 and 13.8.)
//
// Keys at or below a query's threshold go to its candidate slots in HBM as in
// knn_collect.hip.  An unseeded pass first bounds each query's M-th smallest
// key by bisection over the 192 keys of the first pool tile, which the lane
// pair holds in registers.
#include "collect_device.hpp"

#include <algorithm>

namespace gtann {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));   // a value: never memory

constexpr int kSplitChunk = 32;   // dimensions per chunk
constexpr int kSplitRows = 192;   // pool rows per tile: six accumulators per wave
constexpr int kSplitTiles = kSplitRows / kPoolTile;
constexpr int kRowPieces = kSplitChunk / 4;            // 16-byte pieces of a row's chunk in the copy: 4 floats
constexpr int kTilePieces = 3 * kSplitChunk / 8;       // and in LDS: 8 h of each quarter, then m, then l

// Where the copy of the rows holds piece 0 of chunk 0 of the row at position
// p, in pieces: groups of 32 positions, chunk-major, a chunk's pieces one
// after another, each for the group's 32 rows.  A tile's chunk is then a few
// whole 4 KiB blocks, and 32 lanes with consecutive rows read 512 consecutive
// bytes.
__device__ __forceinline__ uint32_t piece_at(uint32_t p, int nch)
{
    return (p >> 5) * static_cast<uint32_t>(nch * kRowPieces * 32) + (p & 31u);
}

// The rows X[members[p]] (stride Dp; members null: X[p]), scaled, to Xs at
// their positions p; ex[p] = -k.  *bad is set by rows that the inner product
// cannot take.  One block per 32 positions, eight lanes per row.
__global__ void __launch_bounds__(256) split_rows_kernel(const float* __restrict__ X, const float* __restrict__ nrm,
                                                         const int32_t* __restrict__ members, int64_t N, int Dp,
                                                         f32x4* __restrict__ Xs, int32_t* __restrict__ ex,
                                                         unsigned int* __restrict__ bad)
{
    const int piece = threadIdx.x & 7;
    const int64_t pos = static_cast<int64_t>(blockIdx.x) * 32 + (threadIdx.x >> 3);
    if (pos >= N) return;
    const int64_t row = members ? members[pos] : pos;
    const f32x4* x = reinterpret_cast<const f32x4*>(X + row * Dp) + piece;
    const float n = nrm[row];
    const bool finite = n < INFINITY;
    // |x| < 2^e; norms too small to be exact: every element is below 2^-50
    int e = -50;
    if (finite && n >= 0x1p-100f) frexpf(sqrtf(n), &e);
    const int k = finite ? 57 - e : 0;
    const int nch = Dp / kSplitChunk;
    f32x4* out = Xs + piece_at(static_cast<uint32_t>(pos), nch) + piece * 32;
    bool tiny = !finite;
    constexpr int U = 4;
    for (int c0 = 0; c0 < nch; c0 += U) {
        f32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = x[kRowPieces * min(c0 + u, nch - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c0 + u >= nch) break;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[u][i] = finite ? ldexpf(v[u][i], k) : 0.f;
                tiny = tiny || (v[u][i] != 0.f && fabsf(v[u][i]) < 0x1p-48f);
            }
            out[(c0 + u) * kRowPieces * 32] = v[u];
        }
    }
    if (piece == 0) ex[pos] = -k;
    if (__ballot(tiny) && (threadIdx.x & 63) == 0) atomicOr(bad, 1u);
}

__global__ void split_clear_kernel(unsigned int* bad) { *bad = 0u; }

// Bytes of the copy of n rows
size_t split_copy_bytes(int64_t n, int Dp)
{
    return static_cast<size_t>(ceil_div(n, int64_t(32)) * 32) * Dp * sizeof(float);
}

void launch_split_rows(const float* X, const float* nrm, const int32_t* members, int64_t N, int Dp, float* Xs,
                       int32_t* ex, unsigned int* bad, hipStream_t s)
{
    GT_REQUIRE(Dp % kSplitChunk == 0 && Dp <= 1024 && split_copy_bytes(N, Dp) <= size_t(16) << 32, "split rows: sizes");
    hipLaunchKernelGGL(split_clear_kernel, dim3(1), dim3(1), 0, s, bad);
    if (N > 0)
        hipLaunchKernelGGL(split_rows_kernel, dim3(static_cast<unsigned>(ceil_div(N, int64_t(32)))), dim3(256), 0, s, X,
                           nrm, members, N, Dp, reinterpret_cast<f32x4*>(Xs), ex, bad);
    GT_HIP(hipGetLastError());
}

// Floats as sums of three bf16: h the nearest to it, m the nearest to the
// rest, l what is left; elements 2 i and 2 i + 1 in word i of each part.
__device__ __forceinline__ void split4(const f32x4& z, u32x2 (&part)[3])
{
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        f32x2 r = {z[2 * i], z[2 * i + 1]};
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const uint32_t p = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
            part[x][i] = p;
            r = f32x2{r[0] - __uint_as_float(p << 16), r[1] - __uint_as_float(p & 0xFFFF0000u)};
        }
    }
}

template <int NW>
struct WideCollectSmem {
    __bf16 tile[2][kSplitTiles * kTilePieces * 32 * 8];   // 32-row blocks: a piece's 32 rows one after another
    float tnorm[2][kSplitRows];     // |p|^2 (L2) or 0 (IP); +inf past the slice end
    int32_t tex[2][kSplitRows];     // -k of the row
    int32_t trow[2][kSplitRows];    // pool row id, -1 past the slice end
    CollectWave wv[NW];
};

template <int METRIC, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 8 ? 2 : 1)))
knn_wide_collect_kernel(KnnArgs a, const f32x4* __restrict__ Xs, const int32_t* __restrict__ ex,
                        const f32x4* __restrict__ Qs, const int32_t* __restrict__ qex,
                        const int32_t* __restrict__ p_pos)
{
    extern __shared__ __align__(16) unsigned char smem[];
    using Smem = WideCollectSmem<NW>;
    Smem& sm = *reinterpret_cast<Smem*>(smem);
    constexpr int T = 64 * NW;
    constexpr int PT = kSplitRows * kRowPieces / T;   // pieces of a chunk's rows per thread
    static_assert(PT * T == kSplitRows * kRowPieces && T % 256 == 0 && PT % 3 == 0, "a thread's pieces are of one row and place");

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
    const int64_t qpos = qvalid ? qi : it.q_begin;
    const int qe = qex[qpos];

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

    // thread tid stages piece tid / 32 % 8 of row tid % 32 of the 32-row blocks
    // tid / 256 + T / 256 u (rows past the slice hold the last row's values:
    // their norm is +inf and their id -1)
    const int piece = (tid >> 5) & 7;
    uint32_t at[PT], at_n[PT];   // of this tile and the next: the pieces of chunk 0
    f32x4 pre[PT];
    auto set_at = [&](int stile, uint32_t (&o)[PT]) {
#pragma unroll
        for (int u = 0; u < PT; ++u) {
            const int r = 32 * (tid / 256 + T / 256 * u) + j;
            const int64_t pl = it.p_begin + min(stile * kSplitRows + r, pcount - 1);
            o[u] = piece_at(static_cast<uint32_t>(p_pos ? p_pos[pl] : pl), nch) + 32 * piece;
        }
    };
    auto load_pool = [&](bool next, int c) {
#pragma unroll
        for (int u = 0; u < PT; ++u) pre[u] = Xs[(next ? at_n[u] : at[u]) + static_cast<uint32_t>(c * kRowPieces * 32)];
    };
    auto store_pool = [&](int buf, int u) {
        u32x2 part[3];
        asm volatile("" : "+v"(pre[u]));   // not before here
        split4(pre[u], part);
        u32x2* t = reinterpret_cast<u32x2*>(sm.tile[buf]) + (tid / 256 + T / 256 * u) * (kTilePieces * 64) +
                    (piece >> 1) * 64 + 2 * j + (piece & 1);
#pragma unroll
        for (int x = 0; x < 3; ++x) t[x * 4 * 64] = part[x];
    };
    // the query's chunk: h of dims 8 h.., 16 + 8 h.., then m, then l
    const f32x4* qrow0 = Qs + piece_at(static_cast<uint32_t>(qpos), nch) + 64 * h;
    bf16x8 qc[6];
    f32x4 qx[4];
    auto load_q = [&](int c) {
#pragma unroll
        for (int s = 0; s < 4; ++s) qx[s] = qrow0[static_cast<uint32_t>(c * kRowPieces * 32 + (s >> 1) * 128 + (s & 1) * 32)];
    };
    auto split_q = [&]() {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u32x2 a0[3], a1[3];
            asm volatile("" : "+v"(qx[2 * s]), "+v"(qx[2 * s + 1]));   // not before here
            split4(qx[2 * s], a0);
            split4(qx[2 * s + 1], a1);
#pragma unroll
            for (int x = 0; x < 3; ++x) qc[2 * x + s] = __builtin_bit_cast(bf16x8, u32x4{a0[x][0], a0[x][1], a1[x][0], a1[x][1]});
        }
    };
    // id, norm and scale of tile stile's row tid
    auto tile_meta = [&](int stile, int32_t& id, float& n, int32_t& x) {
        id = -1;
        n = INFINITY;
        x = 0;
        const int p = stile * kSplitRows + tid;
        if (tid < kSplitRows && p < pcount) {
            const int64_t pl = it.p_begin + p;
            id = a.p_rows ? a.p_rows[pl] : static_cast<int32_t>(pl);
            n = METRIC == 0 ? a.np[id] : 0.f;
            x = ex[p_pos ? p_pos[pl] : pl];
        }
    };
    static_assert(T >= kSplitRows, "one row's ids per thread");

    if (nst > 0) {
        set_at(0, at);
        set_at(1, at_n);
        int32_t nrow, nex;
        float nnrm;
        tile_meta(0, nrow, nnrm, nex);
        if (tid < kSplitRows) {
            sm.trow[0][tid] = nrow;
            sm.tnorm[0][tid] = nnrm;
            sm.tex[0][tid] = nex;
        }
        load_pool(false, 0);
        load_q(0);
#pragma unroll
        for (int u = 0; u < PT; ++u) store_pool(0, u);
        split_q();
        __syncthreads();
    }

    int g = 0;
    for (int stile = 0; stile < nst; ++stile) {
        floatx16 acc[kSplitTiles];
#pragma unroll
        for (int u = 0; u < kSplitTiles; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[u][r] = 0.f;
        int32_t nrow, nex;
        float nnrm;
        tile_meta(stile + 1, nrow, nnrm, nex);
#pragma unroll 1
        for (int c = 0; c < nch; ++c) {
            const int buf = g & 1;
            const bool last = c + 1 == nch;
            load_pool(last, last ? 0 : c + 1);
            load_q(last ? 0 : c + 1);
            // the next chunk's loads stay ahead of this chunk's MFMAs
            __builtin_amdgcn_sched_barrier(0);
            // A = pool row u*32 + (lane%32), B = query lane%32.  The h h sums
            // and the smaller products are kept apart and added in fp32
            // instructions, which round to nearest: the matrix cores cut what
            // they add off below the largest term (single products of rows of
            // one element: 0.42 ulps rms with one sum, 0.29 in fp32).  The
            // chunk's sum is added to the running dot, so that the rounding
            // error grows with sqrt(chunks)
#pragma unroll
            for (int u = 0; u < kSplitTiles; ++u) {
                bf16x8 av[6];
#pragma unroll
                for (int s = 0; s < 6; ++s)
                    av[s] = *reinterpret_cast<const bf16x8*>(&sm.tile[buf][8 * (32 * (kTilePieces * u + 2 * s + h) + j)]);
                floatx16 part, top;
#pragma unroll
                for (int r = 0; r < 16; ++r) part[r] = top[r] = 0.f;
                auto product = [&](floatx16& sum, int x, int y) __attribute__((always_inline)) {
                    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[2 * x], qc[2 * y], sum, 0, 0, 0);
                    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[2 * x + 1], qc[2 * y + 1], sum, 0, 0, 0);
                };
                product(part, 2, 0);
                product(part, 0, 2);
                product(part, 1, 1);
                product(part, 1, 0);
                product(part, 0, 1);
                product(top, 0, 0);
                // the next chunk is split while the matrix cores are busy
                if (u >= 2 && u < 5) {
#pragma unroll
                    for (int i = 0; i < PT / 3; ++i) store_pool(buf ^ 1, PT / 3 * (u - 2) + i);
                }
                if (u == 5) split_q();
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[u][r] += top[r] + part[r];
                // the sums of one tile at a time: the compiler would put all
                // six off to the end, in registers that there are not
                asm volatile("" : "+v"(acc[u]));
                __builtin_amdgcn_sched_barrier(0x104);
            }
            __syncthreads();
            ++g;
        }
        if (tid < kSplitRows) {
            sm.trow[(stile + 1) & 1][tid] = nrow;
            sm.tnorm[(stile + 1) & 1][tid] = nnrm;
            sm.tex[(stile + 1) & 1][tid] = nex;
        }
#pragma unroll
        for (int u = 0; u < PT; ++u) at[u] = at_n[u];
        set_at(stile + 2, at_n);

        // the keys, in place: lane (j, h) holds rows 8g + 4h + e of every tile
        const int sb = stile & 1;
#pragma unroll
        for (int u = 0; u < kSplitTiles; ++u)
#pragma unroll
            for (int gg = 0; gg < 4; ++gg) {
                const float4 pn = *reinterpret_cast<const float4*>(&sm.tnorm[sb][kPoolTile * u + 8 * gg + 4 * h]);
                const int4 pe = *reinterpret_cast<const int4*>(&sm.tex[sb][kPoolTile * u + 8 * gg + 4 * h]);
                const float n4[4] = {pn.x, pn.y, pn.z, pn.w};
                const int e4[4] = {pe.x, pe.y, pe.z, pe.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float dot = ldexpf(acc[u][4 * gg + e], qe + e4[e]);
                    acc[u][4 * gg + e] = METRIC == 0 ? fmaf(-2.f, dot, n4[e] + qn) : fmaf(-1.f, dot, n4[e]);
                }
            }
        if (stile == 0 && !a.seed_d) {
            // a bound on the M-th smallest key: bisection between the
            // smallest and the largest of the pair's 192 keys (the query
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

// Queries per block of a launch over n_queries queries: 128 (4 waves) where
// those blocks, of which a CU holds one, make no more than one round, else 256
// (8 waves).  Bucketed passes of 960 dimensions, buckets of 1,000, 128 and 256
// queries per block: 32,000 rows 1.58 and 1.77 ms, 34,000 rows 2.75 and 1.84,
// 60,000 rows 2.83 and 2.25.
int wide_queries_per_block(int64_t n_queries) { return n_queries > int64_t(128) * 256 ? 256 : 128; }

// Xs, ex: the split rows by position; p_pos: the position of every pool-list
// entry (null: itself).  Qs, qex: the split queries, query i (its place in
// a.q_rows) at position i.
void launch_wide_collect(const KnnArgs& a, int qpb, const float* Xs, const int32_t* ex, const float* Qs,
                         const int32_t* qex, const int32_t* p_pos, hipStream_t s)
{
    GT_REQUIRE((p_pos != nullptr) == (a.p_rows != nullptr) && a.n_items % 8 == 0 && a.Dp % kSplitChunk == 0 && a.cand && a.cand_cnt && (qpb == 128 || qpb == 256),
               "wide collect launch");
    if (a.n_items <= 0) return;
    auto go = [&](auto kernel, int waves, size_t lds) {
        GT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(lds)));
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(a.n_items)), dim3(static_cast<unsigned>(64 * waves)), lds, s,
                           a, reinterpret_cast<const f32x4*>(Xs), ex, reinterpret_cast<const f32x4*>(Qs), qex, p_pos);
    };
    auto by_metric = [&](auto nw) {
        constexpr int NW = decltype(nw)::value;
        if (a.metric == 0) go(&knn_wide_collect_kernel<0, NW>, NW, sizeof(WideCollectSmem<NW>));
        else go(&knn_wide_collect_kernel<1, NW>, NW, sizeof(WideCollectSmem<NW>));
    };
    if (qpb == 256) by_metric(std::integral_constant<int, 8>{});
    else by_metric(std::integral_constant<int, 4>{});
    GT_HIP(hipGetLastError());
}

}  // namespace gtann
