// search_kernel.hip -- beam (ef) search over a graph on gfx950.
//
// One wave per query runs the reference's sequential best-first search
// (bd/search.py:20-90, graph_search_single) step for step, with the work of
// each step spread over the 64 lanes:
//   * pop: the candidate with the smallest (distance, id).  The candidates of
//     earlier expansions are scanned in LDS while the rows of this expansion
//     are on their way, and that minimum is then compared with the points
//     just pushed; its graph row is requested as soon as it is known, before
//     the best list is brought up to date;
//   * expand: lane j takes neighbour j of the popped row (rows longer than 64
//     in chunks), drops ids outside [0, N), tests-and-sets the visited set;
//     the new ids move to the first lanes in row order, two lanes (j, j + 32)
//     per new float row: lane j sums the dimensions 0 and 1 mod 4, lane j + 32
//     the dimensions 2 and 3 mod 4 (one fmaf chain each, combined as
//     (s0 + s1) + (s2 + s3): the CPU restatement's order, so the value is bit
//     for bit the same).  (Rows brought in by whole lines and turned through
//     LDS, four lanes per row, took as long for one query and 9.0 instead of
//     7.1 ms for S2's 10,000 at ef 200: 8 KiB more LDS per wave);
//   * best list: new points are applied in row order -- appended while the
//     list is short, then each strictly closer point replaces the first slot
//     holding the maximum (np.argmax), the maximum recomputed by a wave max
//     (DPP) after every replacement.  Lists of up to 256 points live in
//     registers, longer ones in LDS.
// Rows are read as they are stored (float, uint8 or int8, any width), so a
// call touches only the rows that it visits.  Byte rows of up to 256
// dimensions are summed as integers (dot4): every partial sum of the float
// chains is then an integer below 2^24, so both give the same value.
//
// The visited set is a hash table in LDS: buckets of 16 bytes, filled front to
// back, up to 15 tried (0, 1, 3, 6, ... buckets on).  A bucket holds eight
// 16-bit entries where the ids are few enough (the id's bits are mixed by a
// bijection, the bucket number takes the top ones, and the entry keeps the
// others and the number of full buckets passed over, which together name the
// id), else four 32-bit ids.  A query that would fill the table past
// 13/16, or meets 15 full buckets (at that load a few tables in 1,000 with
// 16-bit entries, in 20 with ids; 1.1 to 1.3 buckets are read per id), stops with status 1 and the host runs it again with a
// per-wave bitmap of N bits in HBM.  Candidates that can no longer be popped (distance
// beyond a full best list's maximum) are not stored, and are dropped when the
// array fills; status 2 reports a query whose live candidates still do not
// fit (more than the capacity tie at the maximum), which the host turns into
// an error.
//
// What bounds it: one query is a serial chain of expansions (pop -> graph row
// -> visited set -> rows -> lists) of about 9,000 cycles, most of them
// dependent instructions of a wave alone on its SIMD, so a small batch is
// bound by that chain and a large one by it and the waves that LDS holds
// (S2 at ef 200: 23 KiB each).  Whole calls, with what the version that
// copied the base, kept the best list in LDS, popped by a scan of its own and
// read the visited set from HBM at ef 200 took: one query, 200,003 x 100
// float, ef 64: 0.74 -> 0.29 ms; 1,000 queries, 10^6 x 128 bytes, ef 64:
// 1.36 -> 0.35 ms; 10,000 queries, 10^6 x 128 float, ef 200: 11.2 -> 6.8 ms
// (3.7 TB/s of rows).
#include "gtann_common.hpp"

#include <cfloat>
#include <type_traits>

namespace gtann {

__device__ __forceinline__ int lanes_below(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
}

// set bits of m below bit l (uniform)
__device__ __forceinline__ int lanes_below_at(uint64_t m, int l)
{
    return static_cast<int>(__popcll(m & ((1ull << l) - 1ull)));
}

__device__ __forceinline__ uint32_t readlane_u(uint32_t v, int l)
{
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), l));
}

// The smallest of the lanes' 64-bit keys (uniform): the high words first, the
// low words only among the lanes that tie there.
__device__ __forceinline__ uint64_t wave_min_u64(uint64_t k)
{
    const uint32_t hi = static_cast<uint32_t>(k >> 32);
    const uint32_t mh = wave_extreme_u32<false>(hi);
    const uint64_t tie = __ballot(hi == mh);
    uint32_t ml;
    if ((tie & (tie - 1)) == 0)
        ml = readlane_u(static_cast<uint32_t>(k), __ffsll(static_cast<unsigned long long>(tie)) - 1);
    else
        ml = wave_extreme_u32<false>(hi == mh ? static_cast<uint32_t>(k) : 0xFFFFFFFFu);
    return (static_cast<uint64_t>(mh) << 32) | ml;
}

// Loads of a row that may start at any element
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u4u __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u4a __attribute__((ext_vector_type(4)));

// LDS visited table: eight 16-bit entries per bucket (HALF) or four ids.
// Both steps are straight line for the first bucket; the loops beyond it run
// only when some lane's bucket is full or two lanes met in one word.
template <bool HALF>
struct VisitedTable {
    static constexpr int kProbes = 15;   // a displacement of 15 never occurs: no 16-bit entry is all ones
    uint32_t* tab;      // (buckets, 4) words, free entries all ones
    uint32_t bmask;     // buckets - 1
    int nbits, lbits;   // bits mixed, bits of the bucket number

    // a lane's place in the table: the bucket reached and its words
    struct Cursor {
        uint32_t home, pat;   // home bucket, entry pattern without the displacement (HALF) or the id
        int disp;
        u4a w;
    };

    __device__ __forceinline__ uint32_t pattern(const Cursor& c) const
    {
        return HALF ? (c.pat | static_cast<uint32_t>(c.disp)) * 0x10001u : c.pat;
    }
    __device__ __forceinline__ uint32_t* bucket(const Cursor& c) const
    {
        return tab + 4 * ((c.home + static_cast<uint32_t>(c.disp * (c.disp + 1)) / 2u) & bmask);
    }
    __device__ __forceinline__ bool holds(const Cursor& c) const
    {
        const uint32_t p = pattern(c);
        uint32_t hit = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t t = c.w[i] ^ p;
            if constexpr (HALF) hit |= (t - 0x00010001u) & ~t & 0x80008000u;
            else hit |= t == 0u ? 1u : 0u;
        }
        return hit != 0u;
    }
    __device__ __forceinline__ bool full(const Cursor& c) const
    {
        return HALF ? c.w[3] < 0xFFFF0000u : c.w[3] != 0xFFFFFFFFu;
    }
    // lanes with on walk to the first bucket that holds the id (hit) or has a
    // free entry (!hit); lost: neither within kProbes buckets
    __device__ __forceinline__ void walk(Cursor& c, bool on, bool& hit, bool& lost) const
    {
        c.w = *reinterpret_cast<const u4a*>(bucket(c));
        hit = on && holds(c);
        lost = false;
        bool more = on && !hit && full(c);
        while (__ballot(more)) {
            if (more) {
                ++c.disp;
                lost = c.disp == kProbes;
            }
            more = more && !lost;
            const u4a w = *reinterpret_cast<const u4a*>(bucket(c));
            if (more) {
                c.w = w;
                hit = holds(c);
                more = !hit && full(c);
            }
        }
    }
    __device__ __forceinline__ void find(Cursor& c, uint32_t v, bool on, bool& hit, bool& lost) const
    {
        // a bijection of [0, 2^nbits): odd multiplications and a right xorshift
        const uint32_t m = 0xFFFFFFFFu >> (32 - nbits);
        uint32_t x = (v * 0x9E3779B1u) & m;
        x ^= x >> ((nbits + 1) >> 1);
        x = (x * 0x85EBCA6Bu) & m;
        const int rbits = nbits - lbits;
        c.home = x >> rbits;
        c.pat = HALF ? (x & ((1u << rbits) - 1u)) << 4 : v;
        c.disp = 0;
        walk(c, on, hit, lost);
    }
    // lanes with on insert their id where find left the cursor: isnew, or dup
    // (another lane of this call inserted the same id), or lost
    __device__ __forceinline__ void insert(Cursor& c, bool on, bool& isnew, bool& dup, bool& lost) const
    {
        isnew = dup = false;
        while (__ballot(on)) {
            // the first word with a free entry (buckets fill front to back)
            uint32_t old = c.w[3];
            int i = 3;
#pragma unroll
            for (int k = 2; k >= 0; --k) {
                const bool f = HALF ? c.w[k] >= 0xFFFF0000u : c.w[k] == 0xFFFFFFFFu;
                old = f ? c.w[k] : old;
                i = f ? k : i;
            }
            const uint32_t p = pattern(c);
            uint32_t want = p;
            if constexpr (HALF)
                want = old == 0xFFFFFFFFu ? (p | 0xFFFF0000u) : ((old & 0xFFFFu) | (p & 0xFFFF0000u));
            uint32_t got = ~old;
            if (on) got = atomicCAS(bucket(c) + i, old, want);
            isnew = isnew || (on && got == old);
            on = on && got != old;
            if (__ballot(on)) {
                bool hit, l;
                walk(c, on, hit, l);
                dup = dup || (on && hit);
                lost = lost || (on && l);
                on = on && !hit && !l;
            }
        }
    }
};

// The best list: slot i holds a distance key (f2o) and an id.  R > 0: slots
// R lane .. R lane + R - 1 in registers (the first slot that holds a value is
// then in the first lane that does); R = 0: in LDS.
template <int R>
struct BestList {
    typedef uint32_t vec __attribute__((ext_vector_type(R > 0 ? R : 1)));   // a value: never memory
    vec k, id;
    uint32_t* lk;
    uint32_t* li;

    // lane l's (key, id), l < app, into slot nb + l
    __device__ __forceinline__ void append(int lane, int nb, int app, uint32_t key, uint32_t v)
    {
        if constexpr (R > 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int l = R * lane + r - nb;
                const bool mine = l >= 0 && l < app;
                const uint32_t kk = static_cast<uint32_t>(__shfl(static_cast<int>(key), l & 63));
                const uint32_t vv = static_cast<uint32_t>(__shfl(static_cast<int>(v), l & 63));
                k[r] = mine ? kk : k[r];
                id[r] = mine ? vv : id[r];
            }
        } else {
            if (lane < app) {
                lk[nb + lane] = key;
                li[nb + lane] = v;
            }
            wave_sync();
        }
    }
    __device__ __forceinline__ void put(int lane, int slot, uint32_t key, uint32_t v)
    {
        if constexpr (R > 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const bool mine = slot == R * lane + r;
                k[r] = mine ? key : k[r];
                id[r] = mine ? v : id[r];
            }
        } else {
            if (lane == 0) {
                lk[slot] = key;
                li[slot] = v;
            }
            wave_sync();
        }
    }
    // the largest key of the ef slots and the first slot that holds it (slots
    // of registers from ef on hold 0, below every distance's key)
    __device__ __forceinline__ void worst(int lane, int ef, uint32_t& key, int& slot) const
    {
        uint32_t m = 0;
        int first = 0;
        if constexpr (R > 0) {
            m = k[0];
#pragma unroll
            for (int r = 1; r < R; ++r) {
                first = k[r] > m ? r : first;
                m = max(m, k[r]);
            }
            key = wave_extreme_u32<true>(m);
            const int l = __ffsll(static_cast<unsigned long long>(__ballot(m == key))) - 1;
            slot = R * l + (R > 1 ? __builtin_amdgcn_readlane(first, l) : 0);
        } else {
            for (int i = lane; i < ef; i += 64) {
                const uint32_t x = lk[i];
                first = (x > m || i == lane) ? i : first;
                m = max(m, x);
            }
            key = wave_extreme_u32<true>(m);
            slot = static_cast<int>(wave_extreme_u32<false>(lane < ef && m == key ? static_cast<uint32_t>(first) : 0xFFFFFFFFu));
        }
    }
};

// LDS of one query, in order: candidate keys, visited table, query row, new
// ids, their distances, best list (lists of more than 256 points).
// (the query row padded to whole groups of eight quads)
__host__ __device__ inline int search_query_bytes(int D, int esz) { return (D * esz + 127) / 128 * 128 + 16; }
constexpr int kRowQuads = 32;      // quads of dimensions summed at a time (float rows)
constexpr int kLaneQuads = 16;     // the same with a lane per row

// x of the lane that CTRL names, within a row of 16 lanes
template <int CTRL>
__device__ __forceinline__ int row_lane(int x)
{
    return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false);
}

// VS: the visited set (0 bitmap in HBM, 1 table of 16-bit entries, 2 table of ids)
// LANE: float rows by one lane each, up to 64 at a time, instead of two lanes
// each, up to 32 (search_lane_rows).  A load of 16 bytes per lane instead of 8
// asks the vector cache for half as many lines per row, which bounds many
// queries over long rows; two lanes per row have half of the dependent sums
// and registers for a whole row of 128 in flight, which bounds few.
template <typename T, int R, int VS, bool LANE = false>
__global__ void __attribute__((amdgpu_flat_work_group_size(64, 64), amdgpu_waves_per_eu(3))) graph_search_kernel(SearchArgs a)
{
    constexpr bool INT = !std::is_same<T, float>::value;
    constexpr bool BITMAP = VS == 0;
    extern __shared__ __align__(16) unsigned char smem[];
    uint64_t* ck = reinterpret_cast<uint64_t*>(smem);                       // candidate keys (d, id)
    uint32_t* tab = reinterpret_cast<uint32_t*>(ck + a.CC);                 // visited table
    unsigned char* qb = reinterpret_cast<unsigned char*>(tab + 4 * a.buckets);
    const int qbytes = search_query_bytes(a.D, sizeof(T));
    uint32_t* nid = reinterpret_cast<uint32_t*>(qb + qbytes);               // new ids of an expansion (64)

    const int lane = threadIdx.x;
    const uint32_t N = static_cast<uint32_t>(a.N);
    const int D = a.D;
    uint32_t* bm = BITMAP ? a.bitmap + static_cast<int64_t>(blockIdx.x) * a.bm_words : nullptr;
    VisitedTable<VS == 1> vt;
    vt.tab = tab;
    vt.bmask = static_cast<uint32_t>(a.buckets - 1);
    vt.nbits = a.nbits;
    vt.lbits = a.lbits;
    BestList<R> best;
    float* ndv = reinterpret_cast<float*>(nid + 64);                        // their distances
    best.lk = reinterpret_cast<uint32_t*>(ndv + 64);
    best.li = best.lk + a.efr;
    const T* X = static_cast<const T*>(a.X);

    for (int64_t r = blockIdx.x; r < a.n_run; r += gridDim.x) {
        const int64_t q = a.q_list ? a.q_list[r] : r;
        // the query row, zero padded
        {
            const T* Q = static_cast<const T*>(a.Q) + q * a.ld;
            T* qd = reinterpret_cast<T*>(qb);
            const int n = qbytes / static_cast<int>(sizeof(T));
            for (int k = lane; k < n; k += 64) qd[k] = k < D ? Q[k] : static_cast<T>(0);
        }
        if constexpr (!BITMAP) {
            const u4a ones = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};
            for (int k = lane; k < a.buckets; k += 64) reinterpret_cast<u4a*>(tab)[k] = ones;
        }
        wave_sync();
        // Byte rows: a group of G lanes per row, lane p of it with the 16
        // bytes from 16 p on (a last partial piece: the row's last 16 bytes,
        // those of the piece before it masked out)
        int32_t qq = 0;   // |q|^2
        int G = 1, poff = 0;
        u4a pmask = {0u, 0u, 0u, 0u}, qp = pmask;
        // Float rows: lane j + 32 h with dimensions 2 h, 2 h + 1 mod 4
        const int j = lane & 31, h = lane >> 5;
        if constexpr (INT) {
            for (int k = lane; k < D; k += 64) {
                const int32_t y = reinterpret_cast<const T*>(qb)[k];
                qq += y * y;
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) qq += __shfl_xor(qq, o);
            const int np = (D + 15) / 16;
            while (G < np) G *= 2;
            const int p = lane & (G - 1);
            const int skip = p == np - 1 && D >= 16 ? 16 * np - D : 0;   // bytes of the piece before it
            poff = p < np ? 16 * p - skip : 0;
            if (p < np) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int z = min(max(skip - 4 * e, 0), 4);           // bytes masked in word e
                    pmask[e] = z >= 4 ? 0u : 0xFFFFFFFFu << (8 * z);
                    uint32_t y = 0;
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        y |= static_cast<uint32_t>(qb[min(poff + 4 * e + t, qbytes - 1)]) << (8 * t);
                    qp[e] = y & pmask[e];
                }
            }
        }

        int nb = 0;          // best list length
        int nc = 0;          // candidates
        int nvis = 0;        // visited points
        int st = 0;
        int nexp = 0;
        uint32_t worstk = 0; // key of the maximum of the best list once it holds ef points
        int wpos = 0;        // its first slot
        if constexpr (R > 0) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                best.k[i] = 0;
                best.id[i] = 0;
            }
        }

        // the ids of the first row: the entry points, in order
        uint32_t v = 0xFFFFFFFFu;
        if (a.entries) {
            if (lane < a.n_entry) v = static_cast<uint32_t>(a.entries[q * a.n_entry + lane]);
        } else {
            // n_entry draws per query from a splitmix64 stream, sorted and distinct
            uint32_t x = 0xFFFFFFFFu;
            if (lane < a.n_entry) {
                uint64_t z = a.seed + 0x9E3779B97F4A7C15ull * static_cast<uint64_t>(q * a.n_entry + lane + 1);
                z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
                z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
                z ^= z >> 31;
                x = static_cast<uint32_t>(z % static_cast<uint64_t>(a.N));
            }
            bool firstc = lane < a.n_entry;
            for (int i = 0; i < a.n_entry; ++i) firstc = firstc && !(lane > i && readlane_u(x, i) == x);
            const uint64_t fm = __ballot(firstc);
            int rank = 0;
            for (int i = 0; i < a.n_entry; ++i) rank += ((fm >> i) & 1ull) && readlane_u(x, i) < x ? 1 : 0;
            if (firstc) nid[rank] = x;
            wave_sync();
            if (lane < static_cast<int>(__popcll(fm))) v = nid[lane];
            wave_sync();
        }

        uint64_t held = kNoKey;        // smallest candidate stored before this row's pushes
        int hslot = 0;                 // its slot
        uint64_t fresh = kNoKey;       // smallest key pushed by this row
        int fslot = 0;                 // its slot
        uint32_t nrow = 0xFFFFFFFFu;   // graph row of the smaller of the two, lane j's entry (the first 64)
        auto request_row = [&](uint64_t k) __attribute__((always_inline)) {
            const int64_t u = static_cast<uint32_t>(k);
            nrow = lane < a.deg ? a.graph[u * a.deg + lane] : 0xFFFFFFFFu;
        };
        // the smallest stored candidate and a request for its graph row
        auto scan = [&]() __attribute__((always_inline)) {
            uint64_t mk = kNoKey;
            int ms = 0;
            for (int i = lane; i < nc; i += 256) {   // (the array holds a multiple of 64 keys)
                uint64_t k[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) k[t] = ck[min(i + 64 * t, a.CC - 1)];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (i + 64 * t < nc && k[t] < mk) { mk = k[t]; ms = i + 64 * t; }
            }
            held = wave_min_u64(mk);
            if (held != kNoKey) {
                hslot = __builtin_amdgcn_readlane(ms, __ffsll(static_cast<unsigned long long>(__ballot(mk == held))) - 1);
                request_row(held);
            }
        };

        // Visits the ids held by the lanes in lane order (the reference's
        // loop order); lanes without an id hold 0xFFFFFFFF.  last: no more
        // ids of this row follow (the held candidate is found meanwhile).
        // false = the query stopped (st set).
        auto visit = [&](uint32_t v, bool last) __attribute__((always_inline)) -> bool {
            bool isnew = false;
            if constexpr (BITMAP) {
                bool fresh = v < N;
                for (uint64_t m = __ballot(fresh); m; m &= m - 1) {     // repeats of an earlier lane
                    const int i = __ffsll(static_cast<unsigned long long>(m)) - 1;
                    const uint32_t o = readlane_u(v, i);
                    fresh = fresh && !(lane > i && o == v);
                }
                if (fresh) {
                    const uint32_t bit = 1u << (v & 31u);
                    isnew = (atomicOr(&bm[v >> 5], bit) & bit) == 0u;
                }
            } else {
                typename VisitedTable<VS == 1>::Cursor c;
                const bool in = v < N;
                bool hit, lost, dup;
                vt.find(c, v, in, hit, lost);
                wave_sync();   // every lookup precedes this call's insertions
                const bool mine = in && !hit && !lost;
                vt.insert(c, mine, isnew, dup, lost);
                // ids that another lane of this call inserted: the first copy
                // in lane order is the new point
                for (uint64_t d = __ballot(dup); d; d &= d - 1) {
                    const uint32_t o = readlane_u(v, __ffsll(static_cast<unsigned long long>(d)) - 1);
                    const uint64_t same = __ballot(mine && v == o);
                    if (mine && v == o) isnew = lane == __ffsll(static_cast<unsigned long long>(same)) - 1;
                }
                if (__ballot(lost)) { st = 1; return false; }
            }
            const uint64_t newm = __ballot(isnew);
            const int nn = static_cast<int>(__popcll(newm));
            if (nn == 0) {
                if (last) scan();
                return true;
            }
            nvis += nn;
            if (!BITMAP && nvis > a.vlimit) { st = 1; return false; }

            // the new ids to lanes 0 .. nn - 1, in order
            if (isnew) nid[lanes_below(newm)] = v;
            wave_sync();
            if constexpr (INT) {
                const unsigned char* Xb = reinterpret_cast<const unsigned char*>(X);
                const int gs = 31 - __builtin_clz(G), RP = 64 >> gs;   // rows per load
                const int rg = lane >> gs;
                // four loads in flight; rows past the last read the last one's
                for (int base = 0; base < nn; base += 4 * RP) {
                    u4a x[4];
                    uint32_t ux[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) ux[t] = nid[min(base + t * RP + rg, nn - 1)];
                    if (D >= 16) {
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const u4u w = *reinterpret_cast<const u4u*>(Xb + static_cast<int64_t>(ux[t]) * a.ld + poff);
                            x[t] = u4a{w[0], w[1], w[2], w[3]};
                        }
                    } else {
                        for (int t = 0; t < 4; ++t) {
                            u4a w = {0u, 0u, 0u, 0u};
#pragma unroll
                            for (int k = 0; k < 15; ++k)
                                if (k < D)
                                    w[k >> 2] |= static_cast<uint32_t>(Xb[static_cast<int64_t>(ux[t]) * a.ld + k]) << (8 * (k & 3));
                            x[t] = w;
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (last && base == 0) scan();
                    int32_t v2[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        int32_t xx = 0, xq = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint32_t xe = x[t][e] & pmask[e];
                            if constexpr (std::is_same<T, uint8_t>::value) {
                                xx = static_cast<int32_t>(__builtin_amdgcn_udot4(xe, xe, static_cast<uint32_t>(xx), false));
                                xq = static_cast<int32_t>(__builtin_amdgcn_udot4(xe, qp[e], static_cast<uint32_t>(xq), false));
                            } else {
                                xx = __builtin_amdgcn_sdot4(static_cast<int>(xe), static_cast<int>(xe), xx, false);
                                xq = __builtin_amdgcn_sdot4(static_cast<int>(xe), static_cast<int>(qp[e]), xq, false);
                            }
                        }
                        v2[t] = a.metric == 0 ? xx - 2 * xq : xq;
                    }
                    // over the group: exchanges with lanes l ^ 1, l ^ 2, then mirrored halves
#pragma unroll
                    for (int st2 = 0; st2 < 4; ++st2)
                        if (G > (1 << st2)) {
#pragma unroll
                            for (int t = 0; t < 4; ++t)
                                v2[t] += st2 == 0 ? row_lane<0xB1>(v2[t]) : st2 == 1 ? row_lane<0x4E>(v2[t])
                                       : st2 == 2 ? row_lane<0x141>(v2[t]) : row_lane<0x140>(v2[t]);
                        }
                    if ((lane & (G - 1)) == 0) {
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const float s = static_cast<float>(a.metric == 0 ? v2[t] + qq : v2[t]);
                            if (base + t * RP + rg < nn) ndv[base + t * RP + rg] = a.metric == 0 ? s : -s;
                        }
                    }
                }
            } else if constexpr (LANE) {
                // rows past the last new point are not read (zeros)
                const int n4 = D >> 2;
                const bool on = lane < nn;
                const float* row = X + static_cast<int64_t>(nid[min(lane, nn - 1)]) * a.ld;
                const float* qr = reinterpret_cast<const float*>(qb);
                float s[4] = {0.f, 0.f, 0.f, 0.f};
                auto add = [&](float x, float y, float& acc) __attribute__((always_inline)) {
                    const float t = y - x;
                    acc = a.metric == 0 ? fmaf(t, t, acc) : fmaf(y, x, acc);
                };
                f4u x[kLaneQuads];
#pragma unroll
                for (int k = 0; k < kLaneQuads; ++k) x[k] = f4u{0.f, 0.f, 0.f, 0.f};
                for (int q0 = 0; q0 < n4; q0 += kLaneQuads) {
                    const f4u* xr = reinterpret_cast<const f4u*>(row) + q0;
                    const int n = n4 - q0;
                    if (on) {
                        if (n >= kLaneQuads) {
#pragma unroll
                            for (int k = 0; k < kLaneQuads; ++k) x[k] = xr[k];
                        } else {
#pragma unroll
                            for (int k = 0; k < kLaneQuads; ++k)
                                if (k < n) x[k] = xr[k];
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (last && q0 == 0) scan();
                    const float4* yr = reinterpret_cast<const float4*>(qr) + q0;
#pragma unroll
                    for (int k = 0; k < kLaneQuads; ++k)
                        if (k < n) {
                            const float4 y = yr[k];
                            add(x[k][0], y.x, s[0]);
                            add(x[k][1], y.y, s[1]);
                            add(x[k][2], y.z, s[2]);
                            add(x[k][3], y.w, s[3]);
                        }
                }
                for (int t = 0; t < (D & 3); ++t) {
                    const float v = on ? row[4 * n4 + t] : 0.f;
                    if (t == 0) add(v, qr[4 * n4], s[0]);
                    else if (t == 1) add(v, qr[4 * n4 + 1], s[1]);
                    else add(v, qr[4 * n4 + 2], s[2]);
                }
                const float d = (s[0] + s[1]) + (s[2] + s[3]);
                if (on) ndv[lane] = a.metric == 0 ? d : -d;
            } else {
                const int n4 = D >> 2;
                for (int base = 0; base < nn; base += 32) {
                    const uint32_t u = nid[min(base + j, nn - 1)];
                    const float* row = X + static_cast<int64_t>(u) * a.ld;
                    float sa = 0.f, sb = 0.f;
                    int q0 = 0;
                    do {
                        // every load issued before the first use (one memory
                        // latency for rows of up to 131 dimensions); quads
                        // past the row's end stay zero, as the query's
                        f2u x[kRowQuads];
                        const f2u* xr = reinterpret_cast<const f2u*>(row + 4 * q0 + 2 * h);
                        const int n = n4 - q0;
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            if (8 * g + 8 <= n) {
#pragma unroll
                                for (int k = 8 * g; k < 8 * g + 8; ++k) x[k] = xr[2 * k];
                            } else if (8 * g < n) {
#pragma unroll
                                for (int k = 8 * g; k < 8 * g + 8; ++k) {
                                    x[k] = f2u{0.f, 0.f};
                                    if (k < n) x[k] = xr[2 * k];
                                }
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        if (last && base == 0 && q0 == 0) scan();
                        const float2* yr = reinterpret_cast<const float2*>(reinterpret_cast<const float*>(qb) + 4 * q0 + 2 * h);
                        auto quads = [&](auto add) __attribute__((always_inline)) {
#pragma unroll
                            for (int g = 0; g < 4; ++g)
                                if (8 * g < n) {
                                    float2 y[8];
#pragma unroll
                                    for (int k = 0; k < 8; ++k) y[k] = yr[2 * (8 * g + k)];
                                    if (8 * g + 8 > n) {
#pragma unroll
                                        for (int k = 0; k < 8; ++k)
                                            if (8 * g + k >= n) y[k] = make_float2(0.f, 0.f);   // the last D mod 4 dimensions come after
                                    }
#pragma unroll
                                    for (int k = 0; k < 8; ++k) add(x[8 * g + k], y[k]);
                                }
                        };
                        if (a.metric == 0)
                            quads([&](const f2u& xv, const float2& y) __attribute__((always_inline)) {
                                const float ta = y.x - xv[0], tb = y.y - xv[1];
                                sa = fmaf(ta, ta, sa);
                                sb = fmaf(tb, tb, sb);
                            });
                        else
                            quads([&](const f2u& xv, const float2& y) __attribute__((always_inline)) {
                                sa = fmaf(y.x, xv[0], sa);
                                sb = fmaf(y.y, xv[1], sb);
                            });
                        q0 += kRowQuads;
                    } while (q0 < n4);
                    // the last D mod 4 dimensions
                    if (D & 3) {
                        const float* qr = reinterpret_cast<const float*>(qb);
                        auto add = [&](float x, float y, float acc) __attribute__((always_inline)) -> float {
                            const float t = y - x;
                            return a.metric == 0 ? fmaf(t, t, acc) : fmaf(y, x, acc);
                        };
                        const int t0 = 4 * n4 + 2 * h;
                        if (t0 < D) sa = add(row[t0], qr[t0], sa);
                        if (t0 + 1 < D) sb = add(row[t0 + 1], qr[t0 + 1], sb);
                    }
                    float s = sa + sb;
                    s += __shfl_xor(s, 32);
                    if (h == 0 && base + j < nn) ndv[base + j] = a.metric == 0 ? s : -s;
                }
            }
            wave_sync();

            // lane l < nn: new point l
            const uint32_t u = lane < nn ? nid[lane] : 0u;
            const float dv = lane < nn ? ndv[lane] : 0.f;
            const uint32_t key = f2o(dv);
            const bool full0 = nb >= a.ef;
            const float worst0 = o2f(worstk);
            // candidates: a point beyond a full list's maximum is never popped
            const bool push = lane < nn && !(full0 && dv > worst0);
            const uint64_t pm = __ballot(push);
            const int cnt = static_cast<int>(__popcll(pm));
            if (nc + cnt > a.CC) {
                if (full0) {
                    int out = 0;
                    for (int b0 = 0; b0 < nc; b0 += 64) {
                        const int i = b0 + lane;
                        const uint64_t k = i < nc ? ck[i] : kNoKey;
                        const bool keep = k != kNoKey && o2f(static_cast<uint32_t>(k >> 32)) <= worst0;
                        const uint64_t km = __ballot(keep);
                        wave_sync();
                        if (keep) ck[out + lanes_below(km)] = k;
                        out += static_cast<int>(__popcll(km));
                        wave_sync();
                    }
                    nc = out;
                }
                if (nc + cnt > a.CC) { st = 2; return false; }
                if (last) scan();   // the slots moved
            }
            const uint64_t ckey = push ? (static_cast<uint64_t>(key) << 32) | u : kNoKey;
            if (push) ck[nc + lanes_below(pm)] = ckey;
            nc += cnt;
            if (last && cnt > 0) {
                fresh = wave_min_u64(ckey);
                if (fresh < held) {
                    request_row(fresh);
                    fslot = nc - cnt + lanes_below_at(pm, __ffsll(static_cast<unsigned long long>(__ballot(ckey == fresh))) - 1);
                }
            }

            // best list, in lane order
            const int room = a.ef - nb;
            const int app = min(nn, room);
            if (app > 0) {
                best.append(lane, nb, app, key, u);
                nb += app;
                if (nb == a.ef) best.worst(lane, a.ef, worstk, wpos);
            }
            uint64_t rest = __ballot(lane >= app && lane < nn);
            while (rest) {
                const uint64_t m = rest & __ballot(dv < o2f(worstk));
                if (!m) break;
                const int l = __ffsll(static_cast<unsigned long long>(m)) - 1;
                best.put(lane, wpos, readlane_u(key, l), readlane_u(u, l));
                best.worst(lane, a.ef, worstk, wpos);
                rest &= ~((2ull << l) - 1ull);
            }
            wave_sync();   // nid and ck are read and written by the next row
            return true;
        };

        // entry points, then best-first expansion; cn: the next chunk of the
        // row being expanded
        uint32_t u = 0;
        int cn = a.deg;
        while (visit(v, cn >= a.deg)) {
            if (cn < a.deg) {
                v = cn + lane < a.deg ? a.graph[static_cast<int64_t>(u) * a.deg + cn + lane] : 0xFFFFFFFFu;
                cn += 64;
                continue;
            }
            // the smallest candidate: the one held, or one this row pushed
            const uint64_t m = held < fresh ? held : fresh;
            if (m == kNoKey) break;
            u = static_cast<uint32_t>(m);
            v = nrow;
            if (lane == 0) ck[m == held ? hslot : fslot] = kNoKey;   // taken; dropped when the array fills
            wave_sync();
            if (nb >= a.ef && o2f(static_cast<uint32_t>(m >> 32)) > o2f(worstk)) break;
            ++nexp;
            held = kNoKey;
            fresh = kNoKey;
            cn = 64;
        }

        if (st == 0) {
            // the best list in (distance, slot) order: rank by counting, the
            // distances in LDS (over the candidates)
            float* bd = reinterpret_cast<float*>(ck);
            wave_sync();
            // f(slot, key, id) for this lane's slots below nb
            auto each = [&](auto f) __attribute__((always_inline)) {
                if constexpr (R > 0) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (R * lane + r < nb) f(R * lane + r, best.k[r], best.id[r]);
                } else {
                    for (int i = lane; i < nb; i += 64) f(i, best.lk[i], best.li[i]);
                }
            };
            each([&](int i, uint32_t k, uint32_t) { bd[i] = o2f(k); });
            wave_sync();
            each([&](int i, uint32_t k, uint32_t id) {
                const float di = o2f(k);
                int rk = 0;
                for (int t = 0; t < nb; ++t) {
                    const float dj = bd[t];
                    rk += (dj < di || (dj == di && t < i)) ? 1 : 0;
                }
                if (rk < a.topk) {
                    a.out_ids[q * a.topk + rk] = static_cast<int32_t>(id);
                    a.out_d[q * a.topk + rk] = a.metric == 1 ? -di : di;
                }
            });
            for (int t = nb + lane; t < a.topk; t += 64) {
                a.out_ids[q * a.topk + t] = -1;
                a.out_d[q * a.topk + t] = a.metric == 1 ? -INFINITY : INFINITY;
            }
        }
        if (lane == 0) {
            if (st == 0) {
                atomicAdd(&a.totals->expansions, static_cast<unsigned long long>(nexp));
                atomicAdd(&a.totals->visits, static_cast<unsigned long long>(nvis));
            } else if (st == 1) {
                a.redo[atomicAdd(&a.totals->n_redo, 1u)] = static_cast<int32_t>(q);
            } else {
                atomicMin(&a.totals->overflow, static_cast<uint32_t>(q));
            }
        }
        if constexpr (BITMAP) {
            for (int64_t k = lane; k < a.bm_words; k += 64) bm[k] = 0u;
            __threadfence();
        }
        wave_sync();
    }
}

__global__ void search_totals_init_kernel(SearchTotals* t)
{
    t->expansions = 0;
    t->visits = 0;
    t->n_redo = 0;
    t->overflow = 0xFFFFFFFFu;
}

void launch_search_totals_init(SearchTotals* t, hipStream_t s)
{
    hipLaunchKernelGGL(search_totals_init_kernel, dim3(1), dim3(1), 0, s, t);
    GT_HIP(hipGetLastError());
}

// Whether a launch reads float rows a lane each.  10,000 queries of 10^5 x 960
// (ef 64 / 200), times of two lanes per row and one, degree 16: 10.5 / 28.7 and
// 8.6 / 29.6 ms; 32: 14.7 / 38.8 and 10.2 / 34.1; 48: 21.5 / 52.3 and 13.0 /
// 37.4; x 300, degree 32: 3.5 / 10.3 and 3.7 / 13.6, 48: 5.3 / 17.7 and 5.0 /
// 15.3.  1,000 queries (fewer than SIMDs), x 960, degree 32: 1.66 / 4.2 and
// 2.3 / 6.0, 48: 2.5 / 6.1 and 2.4 / 6.7.
bool search_lane_rows(int64_t queries, int D, int degree, bool floats)
{
    return floats && queries > 1024 && ((D > 448 && degree > 16) || (D > 256 && degree > 32));
}

// LDS bytes of one query of the launch a.
size_t search_query_lds(const SearchArgs& a, int esz)
{
    return static_cast<size_t>(a.CC) * 8 + static_cast<size_t>(a.buckets) * 16 +
           static_cast<size_t>(search_query_bytes(a.D, esz)) + 2 * 64 * 4 +
           (a.ef > 256 ? static_cast<size_t>(a.efr) * 8 : 0);
}

template <typename T>
static void launch_search_t(const SearchArgs& a, unsigned grid, hipStream_t s)
{
    const size_t lds = search_query_lds(a, sizeof(T));
    auto go = [&](auto kernel) {
        if (lds > 65536)
            GT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(lds)));
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(64), lds, s, a);
    };
    if constexpr (std::is_same<T, float>::value) {
        if (a.lane_rows) {
            if (a.buckets == 0) {
                if (a.ef <= 256) go(&graph_search_kernel<T, 4, 0, true>);
                else go(&graph_search_kernel<T, 0, 0, true>);
            } else if (a.half) {
                if (a.ef <= 256) go(&graph_search_kernel<T, 4, 1, true>);
                else go(&graph_search_kernel<T, 0, 1, true>);
            } else {
                if (a.ef <= 256) go(&graph_search_kernel<T, 4, 2, true>);
                else go(&graph_search_kernel<T, 0, 2, true>);
            }
            GT_HIP(hipGetLastError());
            return;
        }
    }
    // the best list in registers where four per lane hold it
    if (a.buckets == 0) {
        if (a.ef <= 256) go(&graph_search_kernel<T, 4, 0>);
        else go(&graph_search_kernel<T, 0, 0>);
    } else if (a.half) {
        if (a.ef <= 64) go(&graph_search_kernel<T, 1, 1>);
        else if (a.ef <= 256) go(&graph_search_kernel<T, 4, 1>);
        else go(&graph_search_kernel<T, 0, 1>);
    } else {
        if (a.ef <= 256) go(&graph_search_kernel<T, 4, 2>);
        else go(&graph_search_kernel<T, 0, 2>);
    }
    GT_HIP(hipGetLastError());
}

void launch_graph_search(const SearchArgs& a, int dtype, int64_t grid, hipStream_t s)
{
    if (a.n_run <= 0) return;
    GT_REQUIRE(a.buckets >= 0 && (a.buckets & (a.buckets - 1)) == 0 && (a.buckets > 0 || a.bitmap), "search: visited set");
    GT_REQUIRE(a.n_entry >= 1 && a.n_entry <= 64, "search: 1 <= entry points <= 64");
    GT_REQUIRE(grid >= 1 && grid <= (int64_t(1) << 31) - 1, "search: grid");
    GT_REQUIRE(a.CC % 64 == 0 && a.efr % 64 == 0 && a.ef >= 1 && a.ef <= a.efr && a.CC >= a.efr + 64, "search: list sizes");
    GT_REQUIRE(dtype == GT_DTYPE_F32 || a.D <= 256, "search: byte rows of at most 256 dimensions");
    const unsigned g = static_cast<unsigned>(grid);
    if (dtype == GT_DTYPE_F32) launch_search_t<float>(a, g, s);
    else if (dtype == GT_DTYPE_U8) launch_search_t<uint8_t>(a, g, s);
    else launch_search_t<int8_t>(a, g, s);
}

}  // namespace gtann
