// gfx950 kernels of the NAM consumer for paired reads.
//
//  k_pair_order   sixteen lanes per NAM list, four lists a wave: each NAM's
//                 position in the reference order is the number of NAMs of the
//                 list with a smaller key, counted against the other lanes of
//                 the row, two NAMs a lane for lists of 17 to 32 (one list in
//                 eight), one a lane of the whole wave for lists of up to 64.
//                 Keys are unique (each NAM's (is_rc, ref_id, query_start,
//                 ref_start) is its own first hit), so counting ranks gives the
//                 one sorted order the reference's quicksort reaches.
//  k_pair_order_long  longer lists, a wave each, against 64-key tiles in LDS.
//                 Lists in canonical order are grouped by (is_rc, ref_id), so a
//                 64-NAM chunk only counts against the groups it spans.
//  k_pair_type    one lane per pair: type, top_dropoff, MAPQ, per-block type
//                 counts.
//  k_type_scatter pair ids grouped by type in id order (the host loop of
//                 step2/main.cu:4641-4646) from the scanned block counts.
//  k_joint_wave   one wave per pair with NAMs on both mates:
//                 get_best_scoring_nam_pairs (step2/main.cu:1719-1830),
//                 including its quicksort, whose order of equal entries is
//                 part of the result; k_joint (one lane per pair) takes the
//                 pairs whose entries exceed the wave kernel's LDS.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "kernels.h"
#include "pairs.h"
#include "wave.h"

namespace gis {

// key of a NAM in the reference order: (is_rc, ref_id) as one ordered word,
// then the diagonal max(0, ref_start - query_start) for mate 2 (0 for mate 1),
// n_hits descending, query_end, query_start, ref_end, ref_start, two to a word
// (unsigned comparisons: signed fields with the top bit flipped)
struct NamKey {
    uint64_t g, dn, q, r;
};

__device__ __forceinline__ uint64_t group_word(const gis_nam &n) {
    return (uint64_t)n.is_rc << 32 | (uint32_t)(n.ref_id ^ (int32_t)0x80000000);
}

__device__ __forceinline__ uint64_t two_signed(int32_t a, int32_t b) {
    return (uint64_t)((uint32_t)a ^ 0x80000000u) << 32 | ((uint32_t)b ^ 0x80000000u);
}

__device__ __forceinline__ NamKey nam_key(const gis_nam &n, bool mate2) {
    return NamKey{group_word(n), two_signed(mate2 ? max(0, n.ref_start - n.query_start) : 0, ~n.n_hits),
                  two_signed(n.query_end, n.query_start), two_signed(n.ref_end, n.ref_start)};
}

__device__ __forceinline__ bool key_less(const NamKey &a, const NamKey &b) {
    if (a.g != b.g) return a.g < b.g;
    if (a.dn != b.dn) return a.dn < b.dn;
    if (a.q != b.q) return a.q < b.q;
    return a.r < b.r;
}

// rank += 1 where the key a of the lane q of the row is less than b: the words as
// one 256-bit number, the borrow of a - b, the broadcast in the subtractions
// themselves (nine instructions; from comparisons the compiler made 35)
template <int q>
__device__ __forceinline__ void count_less(const NamKey &a, const NamKey &b, uint32_t &rank) {
    uint32_t t;
#define WORD(x) (uint32_t)(x), (uint32_t)((x) >> 32)
#define DPP " row_newbcast:%c[q] row_mask:0xf bank_mask:0xf\n\t"
    const uint32_t u[8] = {WORD(a.r), WORD(a.q), WORD(a.dn), WORD(a.g)};
    const uint32_t v[8] = {WORD(b.r), WORD(b.q), WORD(b.dn), WORD(b.g)};
    asm volatile("s_nop 1\n\t"  // (a lane read as the compiler's last write to it ends)
        "v_sub_co_u32_dpp %[t], vcc, %[a0], %[b0]" DPP
        "v_subb_co_u32_dpp %[t], vcc, %[a1], %[b1], vcc" DPP
        "v_subb_co_u32_dpp %[t], vcc, %[a2], %[b2], vcc" DPP
        "v_subb_co_u32_dpp %[t], vcc, %[a3], %[b3], vcc" DPP
        "v_subb_co_u32_dpp %[t], vcc, %[a4], %[b4], vcc" DPP
        "v_subb_co_u32_dpp %[t], vcc, %[a5], %[b5], vcc" DPP
        "v_subb_co_u32_dpp %[t], vcc, %[a6], %[b6], vcc" DPP
        "v_subb_co_u32_dpp %[t], vcc, %[a7], %[b7], vcc" DPP
        "v_addc_co_u32 %[rank], vcc, 0, %[rank], vcc"
        : [t] "=&v"(t), [rank] "+v"(rank)
        : [a0] "v"(u[0]), [a1] "v"(u[1]), [a2] "v"(u[2]), [a3] "v"(u[3]), [a4] "v"(u[4]), [a5] "v"(u[5]),
          [a6] "v"(u[6]), [a7] "v"(u[7]), [b0] "v"(v[0]), [b1] "v"(v[1]), [b2] "v"(v[2]), [b3] "v"(v[3]),
          [b4] "v"(v[4]), [b5] "v"(v[5]), [b6] "v"(v[6]), [b7] "v"(v[7]), [q] "n"(q)
        : "vcc");
#undef DPP
#undef WORD
}

// NAMs q, and with TWO 16 + q, of each row counted against the lanes' keys k0
// (NAM lane) and k1 (NAM 16 + lane); every lane active, keys beyond the lists all
// ones; m is the longest of the rows' lists, 16 at most
template <int q, bool TWO>
__device__ __forceinline__ void rank_rows(const NamKey &k0, const NamKey &k1, uint32_t m, uint32_t &rank0,
                                          uint32_t &rank1) {
    if constexpr (q < 16) {
        if (q >= m) return;
        count_less<q>(k0, k0, rank0);
        if constexpr (TWO) {
            count_less<q>(k0, k1, rank1);
            count_less<q>(k1, k0, rank0);
            count_less<q>(k1, k1, rank1);
        }
        rank_rows<q + 1, TWO>(k0, k1, m, rank0, rank1);
    }
}

constexpr int ORDER_WPB = 4;

// the places of cnt NAMs add up to 0 + 1 + .. + cnt - 1, less one for each two equal
// keys (those have equal places)
__device__ __forceinline__ void places_check(const PairDev &P, uint32_t cnt, uint64_t sum) {
    if (sum != (uint64_t)cnt * (cnt - 1) / 2 && lane_id() == 0) atomicOr(P.err, PAIR_ERR_DUPLICATE);
}

// a list of 33 to 64 NAMs in the lanes of a wave: each lane ranks its NAM against
// every other one read straight from the lanes
__device__ __forceinline__ void order_lanes(const PairDev &P, uint32_t r) {
    const uint32_t lane = lane_id();
    const uint64_t o = P.off[r];
    const uint32_t cnt = (uint32_t)(P.off[r + 1] - o);
    const bool valid = lane < cnt;
    gis_nam mine{};
    NamKey ki{};
    if (valid) {
        mine = P.in[o + lane];
        ki = nam_key(mine, r >= P.n_pairs);
    }
    uint32_t rank = 0;
    for (uint32_t q = 0; q < cnt; q++) {
        const NamKey kj{readlane_u64(ki.g, q), readlane_u64(ki.dn, q), readlane_u64(ki.q, q), readlane_u64(ki.r, q)};
        rank += key_less(kj, ki) ? 1u : 0u;
    }
    if (valid) P.ord[o + rank] = mine;
    places_check(P, cnt, wave_sum_dpp(valid ? rank : 0u));
}

// a longer list by a wave
__device__ __forceinline__ void order_list(const PairDev &P, uint32_t r, NamKey *lk) {
    const uint32_t lane = lane_id();
    const uint64_t o = P.off[r];
    const uint32_t cnt = (uint32_t)(P.off[r + 1] - o);
    const bool mate2 = r >= P.n_pairs;
    const gis_nam *in = P.in + o;
    gis_nam *out = P.ord + o;
    uint64_t places = 0;
    for (uint32_t i0 = 0; i0 < cnt; i0 += 64) {
        const uint32_t i = i0 + lane;
        const bool valid = i < cnt;
        gis_nam mine{};
        NamKey ki{};
        if (valid) {
            mine = in[i];
            ki = nam_key(mine, mate2);
        }
        uint32_t u0 = 0, u1 = cnt;
        if (P.grouped) {
            // the groups this chunk spans: [first index of the first NAM's
            // group, one past the last NAM's group)
            const uint32_t last = min(i0 + 63, cnt - 1);
            const uint64_t gf = group_word(in[i0]), gl = group_word(in[last]);
            uint32_t lo = 0, hi = i0;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (group_word(in[mid]) < gf) lo = mid + 1;
                else hi = mid;
            }
            u0 = lo;
            lo = last + 1;
            hi = cnt;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (group_word(in[mid]) <= gl) lo = mid + 1;
                else hi = mid;
            }
            u1 = lo;
        }
        uint32_t rank = 0;
        for (uint32_t t = u0; t < u1; t += 64) {
            const uint32_t j = t + lane;
            if (j < u1) lk[lane] = nam_key(in[j], mate2);
            wave_sync();
            const uint32_t m = min(64u, u1 - t);
            if (valid) {
                for (uint32_t q = 0; q < m; q++) {
                    const NamKey kj = lk[q];
                    rank += key_less(kj, ki) ? 1u : 0u;
                }
            }
            wave_sync();
        }
        if (valid) {
            out[u0 + rank] = mine;
            places += u0 + rank;
        }
    }
    for (int d = 32; d >= 1; d >>= 1) places += __shfl_xor(places, d, 64);
    places_check(P, cnt, places);
}

// gpu_sort_nams, step2/main.cu:3449-3472 (mate 1: step2/main.cu:2275-2286;
// mate 2: Nam::operator<, step2/my_struct.hpp:54-68). Bound by the latency of a
// wave's loads, offsets then NAMs: four lists share them. (65 536 lists of 7.8
// NAMs on average: 37 us, with a wave to a list 100 us.) A list of 33 to 64 NAMs has
// the whole wave for some microseconds. Longer ones go to k_pair_order_long: their
// time grows with the square of their length, and a wave would take those among its
// four one after the other. A block appends its sixteen lists' with one atomic.
__global__ __launch_bounds__(64 * ORDER_WPB) void k_pair_order(PairDev P) {
    __shared__ uint32_t n_long, at_long;
    const uint32_t wid = uni32(threadIdx.x >> 6), rl = lane_id() & 15;
    const uint32_t n_lists = 2 * P.n_pairs;
    constexpr uint32_t PER_BLOCK = 4 * ORDER_WPB;
    for (uint32_t b0 = PER_BLOCK * blockIdx.x; b0 < n_lists; b0 += PER_BLOCK * gridDim.x) {
        const uint32_t r = b0 + 4 * wid + lane_id() / 16;
        const bool mate2 = r >= P.n_pairs;
        const uint64_t o = P.off[min(r, n_lists)];
        const uint32_t all = (uint32_t)(P.off[min(r + 1, n_lists)] - o);
        const uint32_t cnt = all <= 32 ? all : 0;
        const uint32_t m = wave_max(cnt);
        gis_nam n0{}, n1{};
        if (rl < cnt) n0 = P.in[o + rl];
        if (16 + rl < cnt) n1 = P.in[o + 16 + rl];
        const NamKey none{~0ull, ~0ull, ~0ull, ~0ull};
        const NamKey k0 = rl < cnt ? nam_key(n0, mate2) : none, k1 = 16 + rl < cnt ? nam_key(n1, mate2) : none;
        uint32_t rank0 = 0, rank1 = 0;
        if (m <= 16) rank_rows<0, false>(k0, k1, m, rank0, rank1);
        else rank_rows<0, true>(k0, k1, 16, rank0, rank1);
        uint32_t taken = 0;
        if (rl < cnt) {
            P.ord[o + rank0] = n0;
            taken = 1u << rank0;
        }
        if (16 + rl < cnt) {
            P.ord[o + rank1] = n1;
            taken |= 1u << rank1;
        }
        // equal keys have equal ranks
        if ((uint32_t)__popc(row_or(taken)) != cnt && rl == 0) atomicOr(P.err, PAIR_ERR_DUPLICATE);
        for (uint64_t big = ballot(rl == 0 && all > 32 && all <= 64); big; big &= big - 1)
            order_lanes(P, b0 + 4 * wid + (uint32_t)__builtin_ctzll(big) / 16);
        const bool is_long = all > 64 && rl == 0;
        if (__syncthreads_or(is_long)) {
            if (threadIdx.x == 0) n_long = 0;
            __syncthreads();
            uint32_t at = 0;
            if (is_long) at = atomicAdd(&n_long, 1u);
            __syncthreads();
            if (threadIdx.x == 0) at_long = atomicAdd(P.n_long, n_long);
            __syncthreads();
            if (is_long) P.longs[at_long + at] = r;
            __syncthreads();
        }
    }
}

// the lists that k_pair_order appended, a wave each (128 lists of 1000 NAMs and the
// copies: 3.5 ms, inside k_pair_order 13.4)
__global__ __launch_bounds__(64 * ORDER_WPB) void k_pair_order_long(PairDev P) {
    __shared__ NamKey lk[ORDER_WPB][64];
    const uint32_t n = sload(P.n_long);
    for (uint32_t w = wave_index(ORDER_WPB); w < n; w += gridDim.x * ORDER_WPB)
        order_list(P, uni32(P.longs[w]), lk[threadIdx.x >> 6]);
}

// top_dropoff, step2/main.cu:889-898 (0 for an empty list, which the
// reference never asks for)
__device__ __forceinline__ float top_dropoff(const gis_nam *L, uint32_t c) {
    if (!c) return 0.0f;
    const int nh0 = L[0].n_hits;
    if (nh0 <= 2) return 1.0f;
    if (c > 1) return (float)L[1].n_hits / (float)nh0;
    return 0.0f;
}

// float to int, truncating and saturating (NaN -> 0)
__device__ __forceinline__ int f2i_sat(float x) {
    if (x != x) return 0;
    if (x >= 2147483648.0f) return 2147483647;
    if (x <= -2147483648.0f) return (int)0x80000000;
    return (int)x;
}

// get_mapq(nams, nams[0]), step2/main.cu:900-910; the natural log is the
// correctly rounded float logarithm (log in double rounded to float), and
// the uint8 result wraps a negative value as the reference's return type does
__device__ __forceinline__ uint8_t mapq_of(const gis_nam *L, uint32_t c) {
    if (c <= 1) return 60;
    const float s1 = L[0].score, s2 = L[1].score;
    const double mm = L[0].n_hits / 10.0;
    const float min_matches = (float)(mm < 1.0 ? mm : 1.0);
    const float lg = (float)log((double)s1);
    const float a = 40.0f * (1.0f - __fdiv_rn(s2, s1));
    const float v = __fmul_rn(__fmul_rn(a, min_matches), lg);
    const int u = f2i_sat(v);
    return (uint8_t)(u < 60 ? u : 60);
}

struct PairNam {
    int32_t ref_id, rs, qs, nh;
    uint8_t is_rc;
};

__device__ __forceinline__ PairNam pair_nam(const gis_nam &n) {
    return PairNam{n.ref_id, n.ref_start, n.query_start, n.n_hits, n.is_rc};
}

// is_proper_nam_pair, step2/main.cu:870-887; mu + 10 sigma is one fused
// multiply-add, as the reference's device code computes it
__device__ __forceinline__ bool proper_pair(const PairNam &a, const PairNam &b, float lim) {
    if (a.ref_id != b.ref_id || a.is_rc == b.is_rc) return false;
    const int x = max(0, a.rs - a.qs);
    const int y = max(0, b.rs - b.qs);
    const bool r1_r2 = b.is_rc && x <= y && (float)(y - x) < lim;
    const bool r2_r1 = a.is_rc && y <= x && (float)(x - y) < lim;
    return r1_r2 || r2_r1;
}

__device__ __forceinline__ uint64_t joint_bound(uint32_t c1, uint32_t c2, int mt) {
    if (!c1 || !c2) return 0;
    const uint64_t prod = (uint64_t)c1 * c2;
    const uint64_t first = prod < (uint64_t)(2 * mt + 1) ? prod : (uint64_t)(2 * mt + 1);
    return first + min((uint32_t)mt, c1) + min((uint32_t)mt, c2);
}

// gpu_pre_cal_type, step2/main.cu:3552-3581, with the fresh insert-size
// estimate's mu and sigma
__global__ __launch_bounds__(PAIR_BLOCK) void k_pair_type(PairDev P) {
    __shared__ uint32_t cnt[5];
    if (threadIdx.x < 5) cnt[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t p = blockIdx.x * PAIR_BLOCK + threadIdx.x;
    const uint32_t n = P.n_pairs;
    if (p < n) {
        const uint64_t o1 = P.off[p], o2 = P.off[n + p];
        const uint32_t c1 = (uint32_t)(P.off[p + 1] - o1), c2 = (uint32_t)(P.off[n + p + 1] - o2);
        const gis_nam *A = P.ord + o1, *B = P.ord + o2;
        const float d1 = top_dropoff(A, c1), d2 = top_dropoff(B, c2);
        uint8_t t;
        if (!c1 && !c2) t = 0;
        else if (c1 && !c2) t = 1;
        else if (!c1 && c2) t = 2;
        else if (d1 < P.dropoff && d2 < P.dropoff &&
                 proper_pair(pair_nam(A[0]), pair_nam(B[0]), __builtin_fmaf(10.0f, P.sigma, P.mu)))
            t = 3;
        else t = 4;
        P.types[p] = t;
        P.drop[p] = d1;
        P.drop[n + p] = d2;
        P.mapq[p] = mapq_of(A, c1);
        P.mapq[n + p] = mapq_of(B, c2);
        atomicAdd(&cnt[t], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 5) P.tcnt[threadIdx.x * P.nblk + blockIdx.x] = cnt[threadIdx.x];
}

__global__ __launch_bounds__(PAIR_BLOCK) void k_type_scatter(PairDev P) {
    constexpr int W = PAIR_BLOCK / 64;
    __shared__ uint32_t wc[W][5];
    const uint32_t p = blockIdx.x * PAIR_BLOCK + threadIdx.x;
    const uint32_t wid = threadIdx.x >> 6;
    const int t = p < P.n_pairs ? (int)P.types[p] : -1;
    uint32_t wrank = 0;
    for (int tt = 0; tt < 5; tt++) {
        const uint64_t m = __ballot(t == tt);
        if (t == tt) wrank = mbcnt(m);
        if (lane_id() == 0) wc[wid][tt] = (uint32_t)__popcll(m);
    }
    __syncthreads();
    if (t >= 0) {
        uint32_t before = 0;
        for (uint32_t w = 0; w < wid; w++) before += wc[w][t];
        const uint64_t pos = P.tpos[(uint64_t)t * P.nblk + blockIdx.x] + before + wrank;
        P.tids[pos] = p;
    }
}

// type starts, joint total and error bits to the host's pinned words
__global__ void k_pair_totals(PairDev P) {
    const uint32_t t = threadIdx.x;
    if (t <= 5) P.totals[t] = P.tpos[(uint64_t)t * P.nblk];
    else if (t == 6) P.totals[t] = P.joint ? P.joff[P.n_pairs] : 0;
    else if (t == 7) {
        P.totals[t] = *P.err;
        *P.err = *P.n_long = 0;  // for the next step
    }
}

// where pair p's joint entries are put before their offsets are known: after bounds
// of those of the pairs before it that are linear in their lists' lengths (PairDev),
// which needs no scan and no wait for its total, or after their exact bounds
// (k_joint_bounds)
__device__ __forceinline__ uint64_t joint_place(const PairDev &P, uint32_t p, uint64_t o1, uint64_t o2) {
    if (P.jplace) return P.jplace[p];
    const uint64_t s = o1 + (o2 - P.off[P.n_pairs]);
    return s + (s * P.jmul >> 16) + (uint64_t)p * P.jadd;
}

// exact bounds of the pairs' entries, for joint_place once scanned
__global__ __launch_bounds__(PAIR_BLOCK) void k_joint_bounds(PairDev P) {
    const uint32_t p = blockIdx.x * PAIR_BLOCK + threadIdx.x, n = P.n_pairs;
    if (p >= n) return;
    P.jcnt[p] = (uint32_t)joint_bound((uint32_t)(P.off[p + 1] - P.off[p]), (uint32_t)(P.off[n + p + 1] - P.off[n + p]),
                                      P.max_tries);
}

// an entry's NAM fields that the NamPair comparator reads; an absent NAM is
// Nam{} with ref_start = -1
struct CmpNam {
    float score;
    int32_t qe, qs, re, rs;
    uint8_t is_rc;
};

__device__ __forceinline__ CmpNam cmp_nam(const gis_nam *L, int32_t i) {
    if (i < 0) return CmpNam{0.0f, 0, 0, 0, -1, 0};
    const gis_nam &n = L[i];
    return CmpNam{n.score, n.query_end, n.query_start, n.ref_end, n.ref_start, n.is_rc};
}

// the comparator of step2/main.cu:1790-1828 (strict)
__device__ __forceinline__ bool entry_less(const gis_nam_pair &x, const gis_nam_pair &y, const gis_nam *A,
                                           const gis_nam *B) {
    if (x.score != y.score) return x.score > y.score;
    {
        const CmpNam a = cmp_nam(A, x.i1), b = cmp_nam(A, y.i1);
        if (a.score != b.score) return a.score > b.score;
        if (a.is_rc != b.is_rc) return !a.is_rc;
        if (a.qe != b.qe) return a.qe < b.qe;
        if (a.qs != b.qs) return a.qs < b.qs;
        if (a.re != b.re) return a.re < b.re;
        if (a.rs != b.rs) return a.rs < b.rs;
    }
    const CmpNam a = cmp_nam(B, x.i2), b = cmp_nam(B, y.i2);
    if (a.score != b.score) return a.score > b.score;
    if (a.is_rc != b.is_rc) return !a.is_rc;
    if (a.qe != b.qe) return a.qe < b.qe;
    if (a.qs != b.qs) return a.qs < b.qs;
    if (a.re != b.re) return a.re < b.re;
    return a.rs < b.rs;
}

// quick_sort_iterative, step2/main.cu:317-359: Lomuto partitions around the
// last element. Partitions of disjoint ranges do not interact, so taking the
// smaller part first (the larger one waits on a stack of at most log2 n
// ranges) ends in the same array as the reference's order of ranges. The stacks
// are the caller's (of LOMUTO_STACK words: private arrays took 130 registers of
// the wave kernel for a rare case).
constexpr int LOMUTO_STACK = 24;
__device__ __forceinline__ void lomuto_sort(gis_nam_pair *E, int n, const gis_nam *A, const gis_nam *B, int *st_lo,
                                            int *st_hi) {
    int sp = 0;
    int lo = 0, hi = n - 1;
    for (;;) {
        while (lo < hi) {
            const gis_nam_pair pivot = E[hi];
            int i = lo - 1;
            for (int j = lo; j < hi; j++) {
                const gis_nam_pair ej = E[j];
                if (entry_less(ej, pivot, A, B)) {
                    ++i;
                    E[j] = E[i];
                    E[i] = ej;
                }
            }
            const int p = i + 1;
            E[hi] = E[p];
            E[p] = pivot;
            // ranges of one element are left as they are, like the reference
            const int lsz = p - lo, rsz = hi - p;
            if (lsz <= rsz) {
                if (rsz >= 2) {
                    st_lo[sp] = p + 1;
                    st_hi[sp] = hi;
                    sp++;
                }
                hi = p - 1;
            } else {
                if (lsz >= 2) {
                    st_lo[sp] = lo;
                    st_hi[sp] = p - 1;
                    sp++;
                }
                lo = p + 1;
            }
        }
        if (sp == 0) break;
        sp--;
        lo = st_lo[sp];
        hi = st_hi[sp];
    }
}

constexpr int FLAG_WORDS = PAIR_MAX_TRIES / 32;
constexpr uint32_t JOINT_LDS_CAP = 128;  // entries a pair may have in k_joint_wave
constexpr int FLAG_STRIDE = 2 * FLAG_WORDS + 1;  // odd stride: lanes fall on different banks

// get_best_scoring_nam_pairs, step2/main.cu:1719-1830
__global__ __launch_bounds__(PAIR_BLOCK) void k_joint(PairDev P) {
    __shared__ uint32_t flags[PAIR_BLOCK * FLAG_STRIDE];
    const uint32_t p = blockIdx.x * PAIR_BLOCK + threadIdx.x;
    const uint32_t n = P.n_pairs;
    if (p >= n) return;
    const uint64_t o1 = P.off[p], o2 = P.off[n + p];
    const uint32_t c1 = (uint32_t)(P.off[p + 1] - o1), c2 = (uint32_t)(P.off[n + p + 1] - o2);
    const uint32_t cap = (uint32_t)joint_bound(c1, c2, P.max_tries);
    // bounds within JOINT_LDS_CAP (and pairs without entries) are k_joint_wave's
    if (cap <= JOINT_LDS_CAP) return;
    uint32_t *f1 = flags + threadIdx.x * FLAG_STRIDE, *f2 = f1 + FLAG_WORDS;
    for (int w = 0; w < FLAG_WORDS; w++) f1[w] = f2[w] = 0;
    const gis_nam *A = P.ord + o1, *B = P.ord + o2;
    gis_nam_pair *E = P.jtmp + joint_place(P, p, o1, o2);
    const int mt = P.max_tries;
    const float lim = __builtin_fmaf(10.0f, P.sigma, P.mu);
    uint32_t size = 0;
    bool over = false;
    int best = 0;
    auto push = [&](int sc, int a, int b) {
        if (size < cap) E[size] = gis_nam_pair{sc, a, b};
        else over = true;
        size++;
    };
    for (uint32_t i = 0; i < c1; i++) {
        const PairNam a = pair_nam(A[i]);
        for (uint32_t j = 0; j < c2; j++) {
            const PairNam b = pair_nam(B[j]);
            const int joint = a.nh + b.nh;
            // joint < 0.5 * best in double is 2 joint < best in integers
            if (2 * joint < best || size > (uint32_t)(2 * mt)) break;
            if (proper_pair(a, b, lim)) {
                push(joint, (int)i, (int)j);
                if (i < (uint32_t)mt) f1[i >> 5] |= 1u << (i & 31);
                if (j < (uint32_t)mt) f2[j >> 5] |= 1u << (j & 31);
                best = max(best, joint);
            }
        }
        if (size > (uint32_t)(2 * mt)) break;
    }
    const int best1 = best > 0 ? best : A[0].n_hits;
    const uint32_t lim1 = min(c1, (uint32_t)mt);
    for (uint32_t i = 0; i < lim1; i++) {
        const int nh = A[i].n_hits;
        if (nh < best1 / 2) break;
        if (f1[i >> 5] >> (i & 31) & 1u) continue;
        push(nh, (int)i, -1);
    }
    const int best2 = best > 0 ? best : B[0].n_hits;
    const uint32_t lim2 = min(c2, (uint32_t)mt);
    for (uint32_t i = 0; i < lim2; i++) {
        const int nh = B[i].n_hits;
        if (nh < best2 / 2) break;
        if (f2[i >> 5] >> (i & 31) & 1u) continue;
        push(nh, -1, (int)i);
    }
    if (over) {
        atomicOr(P.err, PAIR_ERR_JOINT);
        P.jcnt[p] = 0;
        return;
    }
    int st_lo[LOMUTO_STACK], st_hi[LOMUTO_STACK];
    lomuto_sort(E, (int)size, A, B, st_lo, st_hi);
    P.jcnt[p] = size;
}

// ---------------------------------------------------------------------------
// get_best_scoring_nam_pairs with one wave per pair (pairs whose entry bound
// fits JOINT_LDS_CAP; max_tries up to 31 always does)
//
// The reference's scan over (i, j) is sequential: at each j of a row i it
// leaves the row when the joint hits fall below half the best pushed so far,
// ends when more than 2 max_tries entries are pushed, and else pushes (i, j) if
// the NAMs form a proper pair. Here, in rows of fewer than 64 cells, the cells of
// all rows are taken in order, 64 at once (longer rows: joint_rows). The running
// best and count change at proper cells only, and few cells are proper: one step
// per proper cell tests the cells of its row up to it that were not tested before
// against the running best and then pushes it or, if one of them fails, drops the
// row. (A row at a time left most lanes idle: lists are of 7.8 NAMs on average.)
// The entries are then sorted by counting smaller ones. For that each list's NAMs
// get their rank under the comparator's NAM part, ties sharing one, so that an
// entry is one word: score, rank, rank. Without equal entries the sorted order is
// unique and equals the reference quicksort's; with equal ones one lane replays
// the quicksort on the entries' ranks. (32 768 pairs, 14% of them with 8 to 41
// proper cells: 62 us, before 282 us.)

constexpr int JOINT_WPB = 4;

// a NAM's part of the NamPair comparator as an ordered number; score descending
// (0 and -0 are equal)
struct CmpKey {
    uint64_t s, q, r;
};

__device__ __forceinline__ CmpKey cmp_key(const CmpNam &n) {
    const uint32_t f = __float_as_uint(n.score == 0.0f ? 0.0f : n.score);
    const uint32_t up = f & 0x80000000u ? ~f : f | 0x80000000u;
    return CmpKey{(uint64_t)~up << 32 | (n.is_rc ? 1u : 0u), two_signed(n.qe, n.qs), two_signed(n.re, n.rs)};
}

__device__ __forceinline__ bool cmp_less(const CmpKey &a, const CmpKey &b) {
    if (a.s != b.s) return a.s < b.s;
    if (a.q != b.q) return a.q < b.q;
    return a.r < b.r;
}

__device__ __forceinline__ bool cmp_eq(const CmpKey &a, const CmpKey &b) {
    return a.s == b.s && a.q == b.q && a.r == b.r;
}

__device__ __forceinline__ CmpKey readlane_key(const CmpKey &k, uint32_t l) {
    return CmpKey{readlane_u64(k.s, l), readlane_u64(k.q, l), readlane_u64(k.r, l)};
}

// score, best first, in the high half of an entry's word
__device__ __forceinline__ uint64_t score_word(int32_t sc) { return (uint64_t)~((uint32_t)sc ^ 0x80000000u) << 32; }

// quick_sort_iterative (step2/main.cu:317-359) on entry indices, K the entries'
// ranks; smaller part first as in lomuto_sort
__device__ __forceinline__ void lomuto_idx(uint8_t *I, int n, const uint8_t *K, int *st_lo, int *st_hi) {
    int sp = 0;
    int lo = 0, hi = n - 1;
    for (;;) {
        while (lo < hi) {
            const uint8_t pv = I[hi];
            int i = lo - 1;
            for (int j = lo; j < hi; j++) {
                const uint8_t ej = I[j];
                if (K[ej] < K[pv]) {
                    ++i;
                    I[j] = I[i];
                    I[i] = ej;
                }
            }
            const int p = i + 1;
            I[hi] = I[p];
            I[p] = pv;
            const int lsz = p - lo, rsz = hi - p;
            if (lsz <= rsz) {
                if (rsz >= 2) {
                    st_lo[sp] = p + 1;
                    st_hi[sp] = hi;
                    sp++;
                }
                hi = p - 1;
            } else {
                if (lsz >= 2) {
                    st_lo[sp] = lo;
                    st_hi[sp] = p - 1;
                    sp++;
                }
                lo = p + 1;
            }
        }
        if (sp == 0) break;
        sp--;
        lo = st_lo[sp];
        hi = st_hi[sp];
    }
}

// the fields of a NAM that decide a proper pair
struct CellNam {
    int32_t ref_id, diag, nh;
    uint32_t is_rc;
};

__device__ __forceinline__ CellNam cell_nam(const gis_nam &n) {
    return CellNam{n.ref_id, max(0, n.ref_start - n.query_start), n.n_hits, n.is_rc};
}

// proper_pair on them
__device__ __forceinline__ bool proper_cell(const CellNam &a, const CellNam &b, float lim) {
    if (a.ref_id != b.ref_id || a.is_rc == b.is_rc) return false;
    return (b.is_rc && a.diag <= b.diag && (float)(b.diag - a.diag) < lim) ||
           (a.is_rc && b.diag <= a.diag && (float)(a.diag - b.diag) < lim);
}

// a wave's LDS for pairs of at most cap entries
struct JointLds {
    gis_nam_pair *E;
    CellNam *cells;  // the two lists' first 64 each
    uint32_t *flags;
    uint8_t *I, *K;  // of entries; first ranks of NAMs, 64 a list
    static __host__ __device__ constexpr uint32_t byte_words(uint32_t cap) { return (cap > 64 ? cap + 3 : 64u) / 4; }
    __device__ JointLds(uint32_t *base, uint32_t cap)
        : E(reinterpret_cast<gis_nam_pair *>(base + 2 * 64 * 4)), cells(reinterpret_cast<CellNam *>(base)),
          flags(base + 2 * 64 * 4 + 3 * cap), I(reinterpret_cast<uint8_t *>(flags + 2 * FLAG_WORDS)),
          K(I + 4 * byte_words(cap)) {}
    static __host__ __device__ constexpr uint32_t words(uint32_t cap) {
        return (2 * 64 * 4 + 3 * cap + 2 * FLAG_WORDS + 2 * byte_words(cap) + 3) & ~3u;
    }
};

// The reference's scan a row at a time, 64 columns each: for rows of 64 cells or more.
// In lists of hundreds of NAMs most cells are never reached: a row is left at the
// first cell whose hits fall below half the best, and rows that fail at their first
// cell are passed over together. a0, b0: the lists' first 64 NAMs in the lanes.
// (100 pairs of a repeat-rich genome, lists of up to 458 NAMs: 0.6 ms, by cells of
// all rows in order 1.5 ms. A pair of 1000 x 1000 NAMs whose rows end at
// their first cell: 0.1 ms, by cells 10.3 ms.)
__device__ __forceinline__ void joint_rows(const gis_nam *A, const gis_nam *B, uint32_t c1, uint32_t c2, int mt,
                                           float lim, CellNam a0, const CellNam &b0, gis_nam_pair *E, uint32_t *f1,
                                           uint32_t *f2, uint32_t &size, int &best) {
    const uint32_t lane = lane_id(), most = 2 * (uint32_t)mt + 1;
    const int first = __builtin_amdgcn_readfirstlane(b0.nh);
    uint32_t rows = 0;  // a0: NAMs rows .. rows + 63 of the first list
    for (uint32_t i = 0; i < c1 && size < most; i++) {
        if (i == rows + 64) {
            rows = i;
            a0 = cell_nam(A[min(i + lane, c1 - 1)]);
        }
        // on to the next row whose first cell does not fail (joint < 0.5 * best in
        // double is 2 joint < best in integers)
        const uint64_t on = ballot(2 * (a0.nh + first) >= best) >> (i - rows);
        i = on ? i + (uint32_t)__builtin_ctzll(on) : rows + 64;
        if (i >= c1) break;
        if (!on) {  // none of these 64
            i--;
            continue;
        }
        const uint32_t l = i - rows;
        const CellNam a{__builtin_amdgcn_readlane(a0.ref_id, (int)l), __builtin_amdgcn_readlane(a0.diag, (int)l),
                        __builtin_amdgcn_readlane(a0.nh, (int)l), readlane_u32(a0.is_rc, l)};
        bool left = false;
        for (uint32_t jc = 0; jc < c2 && !left && size < most; jc += 64) {
            const uint32_t j = jc + lane;
            const bool valid = j < c2;
            CellNam b = b0;
            if (jc && valid) b = cell_nam(B[j]);
            const int joint = a.nh + b.nh;
            uint64_t prop = ballot(valid && proper_cell(a, b, lim)), fail = ballot(valid && 2 * joint < best);
            // the proper cells before the first that fails, one after the other
            for (; prop; prop &= prop - 1) {
                const uint64_t me = prop & (0 - prop);
                if (fail & (me | (me - 1)) || size == most) break;
                if (lane_bit(me)) {
                    E[size] = gis_nam_pair{joint, (int)i, (int)j};
                    if (i < (uint32_t)mt) f1[i >> 5] |= 1u << (i & 31);
                    if (j < (uint32_t)mt) f2[j >> 5] |= 1u << (j & 31);
                }
                size++;
                const int jh = __builtin_amdgcn_readlane(joint, __builtin_ctzll(me));
                if (jh > best) {
                    best = jh;
                    fail = ballot(valid && 2 * joint < best) & ~(me | (me - 1));
                }
            }
            left = fail != 0;
        }
    }
}

// the ranks of a list's c < 64 NAMs and of the absent NAM (at c) under the
// comparator's NAM part; true if a score is a NaN
__device__ __forceinline__ bool rank_nams(const gis_nam *L, uint32_t c, uint8_t *ranks) {
    const uint32_t lane = lane_id();
    const CmpNam n = cmp_nam(L, lane < c ? (int32_t)lane : -1);
    const CmpKey k = cmp_key(n);
    uint32_t rank = 0;
    for (uint32_t q = 0; q <= c; q++) rank += cmp_less(readlane_key(k, q), k) ? 1u : 0u;
    if (lane <= c) ranks[lane] = (uint8_t)rank;
    return ballot(n.score != n.score) != 0;
}

__global__ __launch_bounds__(64 * JOINT_WPB) void k_joint_wave(PairDev P, uint32_t lds_cap) {
    extern __shared__ __align__(16) uint32_t joint_lds[];
    const uint32_t wid = uni32(threadIdx.x >> 6), lane = lane_id();
    const JointLds L(joint_lds + wid * JointLds::words(lds_cap), lds_cap);
    gis_nam_pair *E = L.E;
    CellNam *ca = L.cells, *cb = ca + 64;
    uint32_t *f1 = L.flags, *f2 = f1 + FLAG_WORDS;
    const uint32_t n = P.n_pairs;
    const int mt = P.max_tries;
    const float lim = __builtin_fmaf(10.0f, P.sigma, P.mu);
    for (uint32_t p = wave_index(JOINT_WPB); p < n; p += gridDim.x * JOINT_WPB) {
        const uint64_t o1 = sload(P.off + p), o2 = sload(P.off + n + p);
        const uint32_t c1 = (uint32_t)(sload(P.off + p + 1) - o1), c2 = (uint32_t)(sload(P.off + n + p + 1) - o2);
        const uint64_t cap = joint_bound(c1, c2, mt);
        if (cap == 0 || cap > lds_cap) {
            // no entries, or a bound beyond LDS: k_joint takes the pair
            if (cap == 0 && lane == 0) P.jcnt[p] = 0;
            continue;
        }
        const gis_nam *A = P.ord + o1, *B = P.ord + o2;
        gis_nam_pair *out = P.jtmp + joint_place(P, p, o1, o2);
        // the first 64 NAMs of each list (lane i: NAM i)
        CellNam a0{}, b0{};
        if (lane < c1) ca[lane] = a0 = cell_nam(A[lane]);
        if (lane < c2) cb[lane] = b0 = cell_nam(B[lane]);
        const int nh1 = a0.nh, nh2 = b0.nh;
        if (lane < 2 * FLAG_WORDS) f1[lane] = 0;
        wave_sync();
        const uint32_t most = 2 * (uint32_t)mt + 1;
        uint32_t size = 0;
        int best = 0;
        const uint64_t cells = (uint64_t)c1 * c2;
        // rows of 64 cells or more fill the lanes by themselves
        if (c2 >= 64) joint_rows(A, B, c1, c2, mt, lim, a0, b0, E, f1, f2, size, best);
        // this lane's cell, 64 further on each pass
        uint32_t i = lane / c2, j = lane % c2;
        const uint32_t di = 64 / c2, dj = 64 % c2;
        uint32_t dead = 0xffffffffu;  // the row left last
        for (uint64_t q0 = 0; c2 < 64 && q0 < cells && size < most; q0 += 64) {
            const bool valid = lane < cells - q0;
            bool prop = false;
            int joint = 0;
            if (valid) {
                const CellNam a = i < 64 ? ca[i] : cell_nam(A[i]), b = cb[j];
                joint = a.nh + b.nh;
                prop = proper_cell(a, b, lim);
            }
            // the lanes from this cell's row's first one up to this one
            const uint64_t mine = (2ull << lane) - (1ull << (lane > j ? lane - j : 0));
            uint64_t rem = ballot(prop && i != dead);
            for (;;) {
                // every cell against the best before it if all of rem are pushed
                // (joint < 0.5 * best in double is 2 joint < best in integers)
                int high = best;
                if (rem) high = max(high, wave_excl_max(lane_bit(rem) ? joint : (int)0x80000000));
                const uint64_t fail = ballot(valid && 2 * joint < high);
                // the first one that is not: all before it are
                const uint64_t drop = ballot((fail & mine) != 0) & rem;
                uint64_t push = drop ? rem & ((drop & (0 - drop)) - 1) : rem;
                if (push) {
                    const uint32_t at = size + mbcnt(push);
                    push &= ballot(at < most);
                    int jh = (int)0x80000000;
                    if (lane_bit(push)) {
                        jh = joint;
                        E[at] = gis_nam_pair{joint, (int)i, (int)j};
                        if (i < (uint32_t)mt) atomicOr(&f1[i >> 5], 1u << (i & 31));
                        if (j < (uint32_t)mt) atomicOr(&f2[j >> 5], 1u << (j & 31));
                    }
                    best = max(best, wave_imax(jh));
                    size += (uint32_t)__popcll(push);
                }
                if (!drop || size >= most) {
                    // the last row may go on
                    const uint32_t il = readlane_u32(i, 63);
                    if (fail & ballot(i == il)) dead = il;
                    break;
                }
                dead = readlane_u32(i, (uint32_t)__builtin_ctzll(drop));
                rem &= ballot(i > dead);
            }
            i += di;
            j += dj;
            if (j >= c2) {
                j -= c2;
                i++;
            }
        }
        wave_sync();
        // NAMs of each mate in no pushed pair, while their hits reach half
        // the best joint hits (the list's first NAM's hits without one)
        for (int m = 0; m < 2; m++) {
            const gis_nam *M = m ? B : A;
            const uint32_t c = m ? c2 : c1;
            const uint32_t *fl = m ? f2 : f1;
            const int nh0 = m ? nh2 : nh1;
            const int bestm = best > 0 ? best : __builtin_amdgcn_readfirstlane(nh0);
            const uint32_t lm = min(c, (uint32_t)mt);
            for (uint32_t ic = 0; ic < lm; ic += 64) {
                const uint32_t k = ic + lane;
                const bool valid = k < lm;
                const int nh = !valid ? 0 : (ic == 0 ? nh0 : M[k].n_hits);
                const uint64_t sm = ballot(valid && nh < bestm / 2);
                const uint64_t before = sm ? (sm & (0 - sm)) - 1 : ~0ull;
                const uint64_t qm = ballot(valid && !((fl[k >> 5 & (FLAG_WORDS - 1)] >> (k & 31)) & 1u)) & before;
                if (lane_bit(qm)) E[size + mbcnt(qm)] = m ? gis_nam_pair{nh, -1, (int)k} : gis_nam_pair{nh, (int)k, -1};
                size += (uint32_t)__popcll(qm);
                if (sm) break;
            }
        }
        wave_sync();
        const uint32_t ne = uni32(size);
        if (lane == 0) P.jcnt[p] = ne;
        if (ne <= 1) {  // (most pairs)
            if (lane < ne) out[0] = E[0];
            wave_sync();
            continue;
        }
        uint32_t rank[2] = {0, 0};
        bool tie = false, nan = false;
        if (c1 < 64 && c2 < 64) {
            nan = rank_nams(A, c1, L.I);
            nan |= rank_nams(B, c2, L.K);
            wave_sync();
            uint64_t w[2] = {0, 0};
            for (int k = 0; k < 2; k++) {
                const uint32_t e = lane + 64 * k;
                if (e >= ne) continue;
                const gis_nam_pair x = E[e];
                w[k] = score_word(x.score) | (uint32_t)L.I[x.i1 < 0 ? c1 : (uint32_t)x.i1] << 8 |
                       L.K[x.i2 < 0 ? c2 : (uint32_t)x.i2];
            }
            for (uint32_t f = 0; f < ne; f++) {
                const uint64_t o = f < 64 ? readlane_u64(w[0], f) : readlane_u64(w[1], f - 64);
                rank[0] += o < w[0] ? 1u : 0u;
                tie |= o == w[0] && f != lane && lane < ne;
                if (ne > 64) {
                    rank[1] += o < w[1] ? 1u : 0u;
                    tie |= o == w[1] && f != lane + 64 && lane + 64 < ne;
                }
            }
        } else {
#pragma unroll 1
            for (int k = 0; k < 2; k++) {
                const uint32_t e = lane + 64 * k;
                if (64u * k >= ne) break;
                const gis_nam_pair x = e < ne ? E[e] : gis_nam_pair{0, -1, -1};
                const CmpNam na = cmp_nam(A, x.i1), nb = cmp_nam(B, x.i2);
                const CmpKey xa = cmp_key(na), xb = cmp_key(nb);
                nan |= ballot(na.score != na.score || nb.score != nb.score) != 0;
#pragma unroll 1
                for (uint32_t f0 = 0; f0 < ne; f0 += 64) {
                    const gis_nam_pair y = f0 + lane < ne ? E[f0 + lane] : gis_nam_pair{0, -1, -1};
                    const CmpKey ya = cmp_key(cmp_nam(A, y.i1)), yb = cmp_key(cmp_nam(B, y.i2));
#pragma unroll 1
                    for (uint32_t f = 0; f < min(64u, ne - f0); f++) {
                        const int sc = __builtin_amdgcn_readlane(y.score, (int)f);
                        const CmpKey oa = readlane_key(ya, f), ob = readlane_key(yb, f);
                        const bool eq_s = sc == x.score, eq_a = eq_s && cmp_eq(oa, xa);
                        const bool less = sc > x.score || (eq_s && cmp_less(oa, xa)) || (eq_a && cmp_less(ob, xb));
                        if (less) (k ? rank[1] : rank[0])++;
                        tie |= eq_a && cmp_eq(ob, xb) && f0 + f != e && e < ne;
                    }
                }
            }
        }
        const bool replay = ballot(tie) != 0 && !nan;
        int *stack = reinterpret_cast<int *>(L.cells);
        wave_sync();
        if (nan) {  // no order: the reference's own steps
            if (lane == 0) lomuto_sort(E, (int)ne, A, B, stack, stack + LOMUTO_STACK);
        } else if (replay) {
            for (uint32_t e = lane; e < ne; e += 64) {
                L.I[e] = (uint8_t)e;
                L.K[e] = (uint8_t)(e < 64 ? rank[0] : rank[1]);
            }
            wave_sync();
            if (lane == 0) lomuto_idx(L.I, (int)ne, L.K, stack, stack + LOMUTO_STACK);
        }
        wave_sync();
        for (int k = 0; k < 2; k++) {
            const uint32_t e = lane + 64 * k;
            if (e >= ne) break;
            if (nan) out[e] = E[e];
            else if (replay) out[e] = E[L.I[e]];
            else out[rank[k]] = E[e];
        }
        wave_sync();
    }
}

__global__ __launch_bounds__(PAIR_BLOCK) void k_joint_compact(PairDev P) {
    const uint32_t p = blockIdx.x * PAIR_BLOCK + threadIdx.x;
    if (p >= P.n_pairs) return;
    // (the host sees the total and asks again with room for it)
    if (P.joff[P.n_pairs] > P.jout_cap) return;
    const uint32_t c = P.jcnt[p];
    const gis_nam_pair *src = P.jtmp + joint_place(P, p, P.off[p], P.off[P.n_pairs + p]);
    gis_nam_pair *dst = P.jout + P.joff[p];
    for (uint32_t k = 0; k < c; k++) dst[k] = src[k];
}

size_t pair_blocks(uint32_t n_pairs) { return ((size_t)n_pairs + PAIR_BLOCK - 1) / PAIR_BLOCK; }

void launch_pairs_classify(const PairDev &P, uint64_t *scan_tmp, hipStream_t st) {
    const uint32_t n_lists = 2 * P.n_pairs;
    if (n_lists) {
        const unsigned g = (unsigned)std::min<uint64_t>(((uint64_t)n_lists + 4 * ORDER_WPB - 1) / (4 * ORDER_WPB), 65536);
        hipLaunchKernelGGL(k_pair_order, dim3(g), dim3(64 * ORDER_WPB), 0, st, P);
        const unsigned gl = (unsigned)std::min<uint64_t>(((uint64_t)n_lists + ORDER_WPB - 1) / ORDER_WPB, 2048);
        hipLaunchKernelGGL(k_pair_order_long, dim3(gl), dim3(64 * ORDER_WPB), 0, st, P);
    }
    const unsigned nb = (unsigned)pair_blocks(P.n_pairs);
    if (nb) hipLaunchKernelGGL(k_pair_type, dim3(nb), dim3(PAIR_BLOCK), 0, st, P);
    launch_scan(P.tcnt, const_cast<uint64_t *>(P.tpos), 5ull * nb, scan_tmp, st);
    if (nb) hipLaunchKernelGGL(k_type_scatter, dim3(nb), dim3(PAIR_BLOCK), 0, st, P);
}

void launch_joint_bounds(const PairDev &P, uint64_t *place, uint64_t *scan_tmp, hipStream_t st) {
    const unsigned nb = (unsigned)pair_blocks(P.n_pairs);
    if (nb) hipLaunchKernelGGL(k_joint_bounds, dim3(nb), dim3(PAIR_BLOCK), 0, st, P);
    launch_scan(P.jcnt, place, P.n_pairs, scan_tmp, st);
}

void launch_pairs_joint(const PairDev &P, uint64_t *scan_tmp, hipStream_t st) {
    const unsigned nb = (unsigned)pair_blocks(P.n_pairs);
    if (P.n_pairs) {
        const unsigned g =
            (unsigned)std::min<uint64_t>(((uint64_t)P.n_pairs + JOINT_WPB - 1) / JOINT_WPB, 65536);
        // (LDS for the largest bound there can be: more waves a CU for few tries)
        const uint32_t cap = std::min<uint32_t>(4u * (uint32_t)P.max_tries + 1, JOINT_LDS_CAP);
        hipLaunchKernelGGL(k_joint_wave, dim3(g), dim3(64 * JOINT_WPB), JOINT_WPB * 4 * JointLds::words(cap), st, P,
                           cap);
    }
    // bounds beyond LDS need max_tries above 31
    if (nb && 4u * (uint32_t)P.max_tries + 1 > JOINT_LDS_CAP)
        hipLaunchKernelGGL(k_joint, dim3(nb), dim3(PAIR_BLOCK), 0, st, P);
    launch_scan(P.jcnt, const_cast<uint64_t *>(P.joff), P.n_pairs, scan_tmp, st);
    launch_pairs_joint_compact(P, st);
}

void launch_pairs_joint_compact(const PairDev &P, hipStream_t st) {
    const unsigned nb = (unsigned)pair_blocks(P.n_pairs);
    if (nb) hipLaunchKernelGGL(k_joint_compact, dim3(nb), dim3(PAIR_BLOCK), 0, st, P);
}

void launch_pairs_totals(const PairDev &P, hipStream_t st) {
    hipLaunchKernelGGL(k_pair_totals, dim3(1), dim3(64), 0, st, P);
}

}  // namespace gis
