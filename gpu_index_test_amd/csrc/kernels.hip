// gfx950 kernels of the strobealign seeding path.
//
// One wavefront (64 lanes) owns one read in every per-read kernel. Lanes
// work on positions, windows, seeds or hits of that read in parallel and the
// wave synchronises through LDS or through its own scratch regions. Reads are
// independent: variable-size per-read outputs are placed by scans of per-read
// counts, and waves only meet in the fused kernel's spill list, whose order
// never changes a read's result.
//
// Two forms share the device functions below:
//  - per-stage: k_seed -> k_lookup -> k_hits (reads with many hits, rescued
//    reads) -> k_merge4 -> k_merge -> k_scan_tiles -> k_compact;
//  - fused: k_fused runs the whole path of a read in one wave out of LDS and
//    hands reads that do not fit its LDS budget (long reads, many seeds,
//    many hits) to the per-stage kernels through the spill list.
// Both end in a scan of the per-read NAM counts and k_compact. A launch that
// finds nothing to do still takes ~4.5 us of a batch's run, so the passes over
// few reads share launches, and lists of reads are appended by the kernels that
// decide them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"
#include "seed_dev.h"
#include "wave.h"

namespace gis {

// Lists of reads for the passes over few of them, in DevBatch::sel_ids:
// rescued reads, reads the four-per-wave merge hands on, and reads whose hits
// go to the pool
enum { SEL_RESCUED = 0, SEL_DEFERRED = 1, SEL_POOLED = 2 };

// wave-uniform iteration over a ReadSet
__device__ __forceinline__ uint32_t set_count(const ReadSet &s) { return s.ids ? *s.n_dev : s.n; }
__device__ __forceinline__ uint32_t set_at(const ReadSet &s, uint32_t w) { return s.ids ? s.ids[w] : w; }

// ---------------------------------------------------------------------------
// seeding: canonical syncmers and query randstrobes of one read

struct SeedBufs {
    uint64_t *pk;       // bases 2 bits each, LSB first: base i at bits 2(i%32) of pk[i/32]
    uint8_t *st;        // per k-mer window: anchor state / ST_UNKNOWN / ST_INVALID
    uint64_t *sh;       // canonical s-mer hash per s-mer start
    uint64_t *sy_hash;  // syncmer list (written when sh is done with: may be the same memory)
    uint16_t *sy_pos;   // read positions fit 16 bits (reads are at most 65535 bp)
    uint64_t *nmask;    // bit i set when base i is not ACGT
};

// k-mer hashes over a compacted syncmer list (xxh64 of the canonical k-mer)
__device__ __forceinline__ void syncmer_hashes(uint32_t nh, const SeedParams &P, const SeedBufs &B,
                                               uint64_t *out_sy_hash) {
    for (uint32_t i0 = 0; i0 < nh; i0 += 64) {
        const uint32_t i = i0 + lane_id();
        if (i < nh) {
            const uint64_t hk = xxh64_u64(canonical_code(B.pk, (int)B.sy_pos[i], P.k, P.kmask));
            B.sy_hash[i] = hk;
            if (out_sy_hash) out_sy_hash[i] = hk;
        }
    }
    wave_sync();
}

// canonical s-mer hash at base j (step2/randstrobes.cu:23-32); an s-mer of at
// most 16 bases is a 32-bit code
__device__ __forceinline__ uint64_t smer_hash(const SeedBufs &B, int j, const SeedParams &P) {
    return P.s <= 16 ? xxh64_u64((uint64_t)canonical_code32(B.pk, j, P.s, (uint32_t)P.smask))
                     : xxh64_u64(canonical_code(B.pk, j, P.s, P.smask));
}

// The syncmer scan of a read without N, from the high words of the s-mer
// hashes. A window's state is always a position of its minimum (gis_core.h),
// so the window is a syncmer when the hash at offset t - 1 lies below its
// other w - 1 hashes and is none when it lies above their minimum, whatever
// came before. The high words decide both; where they tie (equal s-mers in
// one window, or a chance of 2^-32 a window) the answer needs the full hashes
// and the windows before: the scan returns false, and the read takes
// syncmer_passes.
__device__ __forceinline__ bool syncmer_fast(int L, const SeedParams &P, const SeedBufs &B, uint32_t cap,
                                             uint64_t *out_sy_pos, uint32_t &nsync) {
    const int lane = (int)lane_id();
    uint32_t *hi = reinterpret_cast<uint32_t *>(B.sh);
    const int ns = L - P.s + 1;
    for (int j0 = 0; j0 < ns; j0 += 64) {
        const int j = j0 + lane;
        if (j < ns) hi[j] = (uint32_t)(smer_hash(B, j, P) >> 32);
    }
    wave_sync();
    const int nk = L - P.k + 1, mid = P.t - 1;
    uint32_t n = 0;
    for (int p0 = 0; p0 < nk; p0 += 64) {
        const int p = p0 + lane;
        bool is_sync = false, tie = false;
        if (p < nk) {
            const uint32_t h = hi[p + mid];
            uint32_t m = 0xffffffffu;
            if (P.w == 5 && mid == 2) {  // every read-length profile up to 375 bp
                m = min(min(hi[p], hi[p + 1]), min(hi[p + 3], hi[p + 4]));
            } else {
                for (int o = 0; o < P.w; o++)
                    if (o != mid) m = min(m, hi[p + o]);
            }
            is_sync = h < m;
            tie = h == m;
        }
        if (ballot(tie)) return false;
        const uint64_t bal = ballot(is_sync);
        if (is_sync) {
            const uint32_t idx = n + mbcnt(bal);
            if (idx < cap) B.sy_pos[idx] = (uint16_t)p;
            if (out_sy_pos) out_sy_pos[idx] = (uint64_t)p;
        }
        n += (uint32_t)__popcll(bal);
    }
    wave_sync();
    nsync = n;
    return true;
}

// What window p does to the state before it (slide, gis_core.h), w <= 7: nibble r is
// the state after state r, nibble 7 and value 7 stand for NONE. st: the window's
// state if it needs no history.
__device__ __forceinline__ uint32_t window_map(const uint64_t *h, int p, int w, uint8_t st) {
    if (st != ST_UNKNOWN) return 0x11111111u * (st < (uint8_t)w ? st : 7u);
    const uint64_t v = h[p + w - 1];
    uint32_t best = (uint32_t)w - 1;
    uint64_t bv = v;
    for (int o = w - 2; o >= 0; o--) {
        const uint64_t c = h[p + o];
        if (c < bv) { bv = c; best = (uint32_t)o; }
    }
    uint32_t m = best | (v < UINT64_MAX ? (uint32_t)w - 1 : 7u) << 28;
    for (int r = 1; r < w; r++) m |= (v < h[p - 1 + r] ? (uint32_t)w - 1 : (uint32_t)r - 1) << (4 * r);
    return m;
}

// the map `first` and then `then`
__device__ __forceinline__ uint32_t map_after(uint32_t then, uint32_t first) {
    uint32_t m = 0;
#pragma unroll
    for (int r = 0; r < 8; r++) m |= (then >> (4 * (first >> (4 * r) & 7u)) & 7u) << (4 * r);
    return m;
}

// The passes of the syncmer scan after packing, for any read: canonical s-mer
// hashes, window states, tie replay and compaction.
__device__ __forceinline__ uint32_t syncmer_passes(int L, const SeedParams &P, const SeedBufs &B, uint32_t cap,
                                                   uint64_t *out_sy_pos) {
    const int lane = (int)lane_id();
    const int k = P.k, s = P.s, w = P.w;

    const int ns = L - s + 1;
    for (int j0 = 0; j0 < ns; j0 += 64) {
        const int j = j0 + lane;
        if (j < ns) B.sh[j] = any_n(B.nmask, j, j + s - 1) ? 0 : smer_hash(B, j, P);
    }
    wave_sync();

    // window states that need no history
    const int nk = L - k + 1;
    for (int p0 = 0; p0 < nk; p0 += 64) {
        const int p = p0 + lane;
        if (p < nk) {
            uint8_t st;
            if (any_n(B.nmask, p, p + k - 1)) {
                st = ST_INVALID;
            } else {
                const bool seg_first = (p == 0) || ((B.nmask[(p - 1) >> 6] >> ((p - 1) & 63)) & 1);
                st = w == 5 ? anchor_state_w<5>(B.sh, p, seg_first) : anchor_state(B.sh, p, w, seg_first);
            }
            B.st[p] = st;
        }
    }
    wave_sync();

    // resolve tied windows from the nearest anchor and compact syncmer
    // positions; a window is a syncmer when its minimum sits at offset t-1
    // (step2/randstrobes.cu:64-69)
    uint32_t nsync = 0;
    uint32_t carry = 7;  // the state of the window before the 64 (w <= 7)
    for (int p0 = 0; p0 < nk; p0 += 64) {
        const int p = p0 + lane;
        uint8_t st = p < nk ? B.st[p] : ST_INVALID;
        const bool tied = ballot(st == ST_UNKNOWN) != 0;
        if (tied && w <= 7) {
            // a tandem repeat ties window after window: the windows' maps
            // composed over the lanes give every state at once. (Each lane
            // walking back by itself was the last waves' time: 100 003 reads of
            // a repeat-rich genome 158 us, now 104.)
            uint32_t m = window_map(B.sh, p, w, st);
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t before = (uint32_t)__shfl_up((int)m, d, 64);
                if (lane >= d) m = map_after(m, before);
            }
            st = (uint8_t)(m >> (4 * carry) & 7u);
        } else if (st == ST_UNKNOWN) {
            // window p-1 is valid and in the same segment; walk back to the
            // segment's nearest anchor (the segment's first window is one)
            int q = p - 1;
            while (q > 0 && B.st[q] == ST_UNKNOWN) q--;
            uint8_t r = B.st[q];
            if (r != ST_NONE && r >= (uint8_t)w) r = ST_NONE;  // cannot happen; keeps indexing in range
            for (int x = q + 1; x <= p; x++) r = slide(r, B.sh, x, w);
            st = r;
        }
        const bool is_sync = p < nk && st == (uint8_t)(P.t - 1);
        carry = readlane_u32(st < (uint8_t)w ? st : 7u, 63);
        const uint64_t bal = ballot(is_sync);
        if (is_sync) {
            const uint32_t idx = nsync + mbcnt(bal);
            if (idx < cap) B.sy_pos[idx] = (uint16_t)p;
            if (out_sy_pos) out_sy_pos[idx] = (uint64_t)p;
        }
        nsync += (uint32_t)__popcll(bal);
    }
    wave_sync();
    return nsync;
}

// the four bases 4 i .. 4 i + 3 of a read as loaded together (their last bytes
// may lie past the read's end: the sequence array has SEQ_PAD bytes after the
// last read), and the mask of those inside it
__device__ __forceinline__ uint32_t four_bases(const char *__restrict__ seq, int L, int i, uint32_t &inside) {
    const int left = L - 4 * i;
    inside = left >= 4 ? 0xffffffffu : left > 0 ? (1u << (8 * left)) - 1u : 0u;
    uint32_t v = 0;
    if (left > 0) __builtin_memcpy(&v, seq + 4 * i, 4);
    return v;
}

// A read's bases packed 2 bits each, four a lane and so 256 a pass: a lane's four
// codes are one byte of the packed array, which is written up to its pad word
// (windows ending in the last word read it). True if every base is ACGT.
__device__ __forceinline__ bool pack_bases(const char *__restrict__ seq, int L, uint64_t *pk) {
    const int nch = (L + 63) >> 6, nbytes = 8 * (2 * nch + 1);
    uint8_t *pkb = reinterpret_cast<uint8_t *>(pk);
    uint32_t any = 0;
    for (int i0 = 0; i0 < nbytes; i0 += 64) {
        const int i = i0 + (int)lane_id();
        uint32_t inside, bad;
        const uint32_t v = four_bases(seq, L, i, inside);
        const uint32_t c = nt4x4(v, bad) & inside;
        any |= bad & inside;
        if (i < nbytes) pkb[i] = (uint8_t)pack4(c);
    }
    wave_sync();
    return ballot(any != 0) == 0;
}

// Canonical syncmers of one read (SyncmerIterator, step2/randstrobes.cu:18-79),
// the whole wave working on the same read. The first `cap` syncmers go to
// B.sy_hash/B.sy_pos (and out_sy_* when given); returns the total count.
//
// Bound by VALU issue. Two passes over a read's bases carry it: four bases a
// lane to pack (150 bases in one pass; one base a lane took three passes and
// two 32-bit spreads each), and the window test on high words, in one pass
// with the compaction. 65,536 reads of 150 bp: 101 -> 64 us.
__device__ __forceinline__ uint32_t seed_syncmers(const char *__restrict__ seq, int L,
                                                  const SeedParams &P, const SeedBufs &B,
                                                  uint32_t cap, uint64_t *out_sy_hash,
                                                  uint64_t *out_sy_pos) {
    const int lane = (int)lane_id();
    const int nch = (L + 63) >> 6;
    const bool clean = pack_bases(seq, L, B.pk);
    uint32_t nsync = 0;
    if (!(clean && syncmer_fast(L, P, B, cap, out_sy_pos, nsync))) {
        // the mask of non-ACGT bases (step2/randstrobes.cu:70-76): bit 4 l + b
        // of 16 lanes' words from the ballots of their byte b
        for (int i0 = 0; 4 * i0 < L; i0 += 64) {
            uint32_t inside, bad;
            const uint32_t v = four_bases(seq, L, i0 + lane, inside);
            (void)nt4x4(v, bad);
            bad &= inside;
            uint64_t m = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint64_t bal = ballot(((bad >> (8 * q)) & 0xffu) != 0);
                uint64_t x = lane < 4 ? (bal >> (16 * lane)) & 0xffffull : 0ull;
                x = (x | (x << 24)) & 0x000000ff000000ffull;
                x = (x | (x << 12)) & 0x000f000f000f000full;
                x = (x | (x << 6)) & 0x0303030303030303ull;
                x = (x | (x << 3)) & 0x1111111111111111ull;
                m |= x << q;
            }
            const int word = i0 / 16 + lane;
            if (lane < 4 && word < nch) B.nmask[word] = m;
        }
        wave_sync();
        nsync = syncmer_passes(L, P, B, cap, out_sy_pos);
    }
    syncmer_hashes(nsync < cap ? nsync : cap, P, B, out_sy_hash);
    return nsync;
}

// LDS of a wave that seeds a long read, and the reads it holds: of up to
// LONG_LDS_BASES bases with up to LONG_LDS_SYNC syncmers (one in k - s + 1 bases on
// average: 2200 to 3100 bases). 6.4 KB, given out as 7.5: 21 waves a CU, five a SIMD.
constexpr int LONG_LDS_BASES = 4096;
constexpr uint32_t LONG_LDS_SYNC = 448;
constexpr int LONG_RING = 128;

struct alignas(8) LongLds {
    uint64_t sy_hash[LONG_LDS_SYNC];
    uint64_t pk[2 * (LONG_LDS_BASES / 64) + 1];
    uint32_t hi[LONG_RING], lo[LONG_RING];
    uint16_t sy_pos[LONG_LDS_SYNC];
};

// the hashes in the ring by s-mer start (the last 64 to 128 of them)
struct RingHash {
    const LongLds &S;
    __device__ __forceinline__ uint64_t operator[](int j) const {
        return (uint64_t)S.hi[j % LONG_RING] << 32 | S.lo[j % LONG_RING];
    }
};

// whether the hash in the middle of the window at p is below (true) or equal to
// (tie) the others' minimum, by high words; W > 0: the window's width
template <int W>
__device__ __forceinline__ bool ring_test(const LongLds &S, int p, int w, int mid, bool &tie) {
    const uint32_t h = S.hi[(p + mid) % LONG_RING];
    uint32_t m = 0xffffffffu;
#pragma unroll
    for (int o = 0; o < (W ? W : w); o++) {
        const uint32_t v = S.hi[(p + o) % LONG_RING];
        m = o == mid ? m : min(m, v);
    }
    tie = h == m;
    return h < m;
}

// The canonical syncmers of a long read from LDS, as syncmer_fast finds them: the
// windows are tested as their last s-mer is hashed, so that the hashes live in a
// ring. A tied window is replayed from the nearest one before it whose state needs
// no history, as syncmer_passes does, while the ring holds that. False if it does
// not, or if the read does not fit or has a base other than ACGT: then it takes
// the passes in global scratch. (8191 reads of 400 to 2500 bp: 91 us; with every pass
// in global scratch 179 us, the latency of the longest reads' chains.)
__device__ __forceinline__ bool long_syncmers(const char *__restrict__ seq, int L, const SeedParams &P, LongLds &S,
                                              const SeedBufs &B, uint64_t *out_sy_pos, uint32_t &nsync) {
    if (L > LONG_LDS_BASES || !pack_bases(seq, L, S.pk)) return false;
    const int lane = (int)lane_id(), ns = L - P.s + 1, mid = P.t - 1;
    uint32_t n = 0;
    for (int j0 = 0; j0 < ns; j0 += 64) {
        const int j = j0 + lane, p = j - (P.w - 1);
        if (j < ns) {
            const uint64_t h = smer_hash(B, j, P);
            S.hi[j % LONG_RING] = (uint32_t)(h >> 32);
            S.lo[j % LONG_RING] = (uint32_t)h;
        }
        wave_sync();
        const bool in = j < ns && p >= 0;
        bool is_sync = false, tie = false;
        if (in) {  // (5 and 7 are the widths of the read-length profiles)
            if (P.w == 5) is_sync = ring_test<5>(S, p, 5, mid, tie);
            else if (P.w == 7) is_sync = ring_test<7>(S, p, 7, mid, tie);
            else is_sync = ring_test<0>(S, p, P.w, mid, tie);
        }
        if (ballot(tie)) {
            bool lost = false;
            if (tie) {
                const RingHash H{S};
                const int oldest = max(0, j0 - 64);
                int q = p;
                uint8_t r = anchor_state(H, q, P.w, q == 0);
                while (r == ST_UNKNOWN && q > oldest) {
                    q--;
                    r = anchor_state(H, q, P.w, q == 0);
                }
                lost = r == ST_UNKNOWN;
                if (!lost)
                    for (int x = q + 1; x <= p; x++) r = slide(r, H, x, P.w);
                is_sync = r == (uint8_t)mid;
            }
            if (ballot(lost)) return false;
        }
        const uint64_t bal = ballot(is_sync);
        if (is_sync) {
            const uint32_t idx = n + mbcnt(bal);
            if (idx < LONG_LDS_SYNC) S.sy_pos[idx] = (uint16_t)p;
            if (out_sy_pos) out_sy_pos[idx] = (uint64_t)p;
        }
        n += (uint32_t)__popcll(bal);
        wave_sync();
    }
    nsync = n;
    return n <= LONG_LDS_SYNC;
}

// Randstrobe number j of a read's query list in randstrobes_query order
// (step2/randstrobes.cu:195-241): j < n_fwd is the forward randstrobe of
// strobe1 = syncmer j, j >= n_fwd the reverse-complement one of strobe1 =
// syncmer n - 1 - (j - n_fwd). The two directions share one code path (lanes
// of both run together without divergence): the reverse-complement pass walks
// the syncmer list backwards, and its positions are mirrored, L - k - pos.
// Candidates lie at index offsets w_min..w_max (RandstrobeIterator::get,
// step2/randstrobes.cu:136-159); positions grow with the index, so the
// reference's break at the first candidate beyond max_dist is the same as
// skipping every candidate beyond it.
struct Rs1 {
    uint64_t h;
    uint32_t s, e;
};

__device__ __forceinline__ Rs1 randstrobe_one(const SeedBufs &B, uint32_t n, uint32_t n_fwd, uint32_t j, int L,
                                              const SeedParams &P) {
    const bool rc = j >= n_fwd;
    const uint32_t i = rc ? j - n_fwd : j;
    const uint32_t last = n - 1;
    const uint32_t k = (uint32_t)P.k;
    const uint32_t mirror = (uint32_t)L - k;  // a syncmer starts at most at L - k
    const uint32_t a = rc ? last - i : i;
    const uint32_t p1 = rc ? mirror - B.sy_pos[a] : B.sy_pos[a];
    const uint64_t h1 = B.sy_hash[a];
    // 32-bit arithmetic in the candidate loop: positions are below 2^32, so
    // the limit clamps there; the cost is at most 64; the high halves of the
    // hashes only count when q has high bits (q = 2^c - 1, c = 8 by default)
    const uint64_t maxp64 = (uint64_t)p1 + P.max_dist_u;
    const uint32_t maxp = maxp64 > 0xffffffffull ? 0xffffffffu : (uint32_t)maxp64;
    const uint32_t qlo = (uint32_t)P.q, qhi = (uint32_t)(P.q >> 32);
    const uint32_t h1lo = (uint32_t)h1, h1hi = (uint32_t)(h1 >> 32);
    const uint32_t *hw = reinterpret_cast<const uint32_t *>(B.sy_hash);
    uint32_t best = a, pbest = p1, minv = 0xffffffffu;
#pragma unroll 1
    for (uint32_t d = P.w_min; d <= P.w_max; d++) {
        if (i + d <= last) {
            const uint32_t x = rc ? a - d : a + d;
            uint32_t c = (uint32_t)__popc((h1lo ^ hw[2 * x]) & qlo);
            if (qhi) c += (uint32_t)__popc((h1hi ^ hw[2 * x + 1]) & qhi);
            const uint32_t px = rc ? mirror - B.sy_pos[x] : B.sy_pos[x];
            if (px <= maxp && c < minv) {
                minv = c;
                best = x;
                pbest = px;
            }
        }
    }
    Rs1 o;
    o.h = h1 + B.sy_hash[best];
    o.s = p1;
    o.e = pbest + k;
    return o;
}

// a read's randstrobes from its n syncmers, in randstrobes_query order: forward
// (strobe1 ascending) then reverse complement, one randstrobe per lane. Returns
// their count.
__device__ __forceinline__ uint32_t seed_randstrobes(uint32_t n, int L, const SeedParams &P, const SeedBufs &B,
                                                     uint64_t *rs_hash, uint32_t *rs_span) {
    const uint32_t n_fwd = ((uint32_t)L >= P.w_max && n > P.w_min) ? n - P.w_min : 0;
    const uint32_t nrs = 2 * n_fwd;
    for (uint32_t j0 = 0; j0 < nrs; j0 += 64) {
        const uint32_t j = j0 + lane_id();
        if (j < nrs) {
            const Rs1 o = randstrobe_one(B, n, n_fwd, j, L, P);
            rs_hash[j] = o.h;
            rs_span[j] = span_pack(o.s, o.e);
        }
    }
    return nrs;
}

struct alignas(8) SeedLds {
    uint64_t sh[LMAX_LDS];  // then the syncmers' hashes
    uint64_t nmask[LMAX_LDS / 64 + 2];
    uint64_t pk[2 * (LMAX_LDS / 64) + 1];
    uint16_t sy_pos[LMAX_LDS];
    uint8_t st[LMAX_LDS];
};

__host__ __device__ inline uint64_t align8(uint64_t x) { return (x + 7) & ~7ULL; }

// global scratch layout of a long read (long_bytes() on the host matches it)
__device__ __forceinline__ SeedBufs long_bufs(uint8_t *base, uint64_t L) {
    SeedBufs B;
    B.sh = (uint64_t *)base;
    B.sy_hash = (uint64_t *)(base + 8 * L);
    B.nmask = (uint64_t *)(base + 16 * L);
    B.sy_pos = (uint16_t *)(base + 16 * L + 8 * (L / 64 + 2));
    // the 8 (2 ceil(L / 64) + 1) bytes of packed bases fit the L bytes given to them (L > 320)
    B.pk = (uint64_t *)(base + 16 * L + 8 * (L / 64 + 2) + align8(4 * L));
    B.st = (uint8_t *)B.pk + align8(L);
    return B;
}

// Seeding parameters of the read-length profiles up to 250 bp (k = 20,
// s = 16, t = 3): kernels instantiated with K20 take them as compile-time
// constants, which shortens the seeding code and frees the scalar registers
// that would hold them. The host launches that instantiation when the
// index's parameters match (is_k20_profile).
__device__ __forceinline__ void pin_k20_profile(SeedParams &P) {
    P.k = 20;
    P.s = 16;
    P.t = 3;
    P.w = 5;
    P.kmask = (1ull << 40) - 1;
    P.smask = 0xffffffffull;
}

static inline bool is_k20_profile(const SeedParams &sp) { return sp.k == 20 && sp.s == 16 && sp.t == 3; }

// the control block cleared by the first threads of one block
static_assert(sizeof(DevCtl) % 4 == 0 && sizeof(DevCtl) / 4 <= 64, "one word per lane");
__device__ __forceinline__ void ctl_clear(DevCtl *ctl) {
    if (threadIdx.x < sizeof(DevCtl) / 4) reinterpret_cast<unsigned *>(ctl)[threadIdx.x] = 0;
}

// (long reads' lengths differ: a block would hold four waves' LDS until its
// longest read is done)
static constexpr int seed_wpb(bool long_reads) { return long_reads ? 1 : SEED_WPB; }

template <bool LONG, bool K20>
__global__ __launch_bounds__(64 * seed_wpb(LONG)) __attribute__((amdgpu_waves_per_eu(LONG ? 6 : 8))) void k_seed(DevBatch b, ReadSet set, SeedParams P,
                                                        int want_sy, int reset) {
    if (K20) pin_k20_profile(P);
    if (reset && blockIdx.x == 0) ctl_clear(b.ctl);
    constexpr int W = seed_wpb(LONG);
    __shared__ SeedLds lds[LONG ? 1 : W];
    __shared__ LongLds long_lds[LONG ? W : 1];
    const int wid = (int)uni32(threadIdx.x >> 6);
    const uint32_t cnt = set_count(set);
    for (uint32_t w = wave_index(W); w < cnt; w += gridDim.x * W) {
        const uint32_t r = set.ids ? sload(set.ids + w) : w;
        const int L = (int)sload(b.read_len + r);
        if ((L > LMAX_LDS) != LONG) continue;
        const uint64_t so = want_sy ? sload(b.sy_off + r) : 0;
        uint64_t *osh = want_sy ? b.sy_hash + so : nullptr;
        uint64_t *osp = want_sy ? b.sy_pos + so : nullptr;
        const uint64_t ro = sload(b.rs_off + r);
        const char *seq = b.seqs + sload(b.read_off + r);
        uint32_t nsync = 0, nrs = 0;
        if (LONG) {
            LongLds &S = long_lds[wid];
            const SeedBufs B{S.pk, nullptr, nullptr, S.sy_hash, S.sy_pos, nullptr};
            if (long_syncmers(seq, L, P, S, B, osp, nsync)) {
                syncmer_hashes(nsync, P, B, osh);
                nrs = seed_randstrobes(nsync, L, P, B, b.rs_hash + ro, b.rs_span + ro);
            } else {
                const SeedBufs G = long_bufs(b.long_scratch + sload(b.long_off + r), (uint64_t)L);
                nsync = seed_syncmers(seq, L, P, G, 0xffffffffu, osh, osp);
                nrs = seed_randstrobes(nsync, L, P, G, b.rs_hash + ro, b.rs_span + ro);
            }
        } else {
            SeedLds &S = lds[wid];
            const SeedBufs B{S.pk, S.st, S.sh, S.sh, S.sy_pos, S.nmask};
            nsync = seed_syncmers(seq, L, P, B, 0xffffffffu, osh, osp);
            nrs = seed_randstrobes(nsync, L, P, B, b.rs_hash + ro, b.rs_span + ro);
        }
        if (lane_id() == 0) {
            b.rs_cnt[r] = nrs;
            b.rs_nfwd[r] = nrs / 2;
            if (want_sy) b.sy_cnt[r] = nsync;
        }
        wave_sync_mem();
    }
}

// The seeds of every read from its slots to their dense place (off: scan of the
// reads' counts), as the ABI's records: query randstrobes (24 bytes) or
// syncmers (16 bytes). One wave a read, a lane a 64-bit word, so that the
// stores are whole lines; a read's slots are several times its seeds, and
// copying them to the host and packing there took most of the call (20,011
// reads of 150 bp: 14.9 ms; now bound by the copy of the records).
__device__ __forceinline__ void emit_offset(const DevBatch &b, const uint64_t *off, uint32_t r, uint64_t o,
                                            uint64_t *h_off) {
    h_off[r] = o;
    if (r + 1 == b.n_reads) h_off[r + 1] = sload(off + r + 1);
}

__global__ __launch_bounds__(64 * WPB) void k_emit_randstrobes(DevBatch b, const uint64_t *off, uint64_t *out,
                                                         uint64_t *h_off) {
    for (uint32_t r = wave_index(WPB); r < b.n_reads; r += gridDim.x * WPB) {
        const uint32_t n = sload(b.rs_cnt + r), half = sload(b.rs_nfwd + r);
        const uint64_t base = sload(b.rs_off + r);
        const uint64_t o = sload(off + r);
        uint64_t *dst = out + 3 * o;
        if (h_off && lane_id() == 0) emit_offset(b, off, r, o, h_off);
        for (uint32_t w = lane_id(); w < 3 * n; w += 64) {
            const uint32_t j = w / 3, c = w - 3 * j;
            const uint32_t sp = b.rs_span[base + j];
            const uint64_t h = b.rs_hash[base + j];
            dst[w] = c == 0 ? h : c == 1 ? (uint64_t)span_start(sp) | ((uint64_t)span_end(sp) << 32) : j >= half ? 1u : 0u;
        }
    }
}

__global__ __launch_bounds__(64 * WPB) void k_emit_syncmers(DevBatch b, const uint64_t *off, uint64_t *out,
                                                      uint64_t *h_off) {
    for (uint32_t r = wave_index(WPB); r < b.n_reads; r += gridDim.x * WPB) {
        const uint32_t n = sload(b.sy_cnt + r);
        const uint64_t base = sload(b.sy_off + r);
        const uint64_t o = sload(off + r);
        uint64_t *dst = out + 2 * o;
        if (h_off && lane_id() == 0) emit_offset(b, off, r, o, h_off);
        for (uint32_t w = lane_id(); w < 2 * n; w += 64) dst[w] = (w & 1 ? b.sy_pos : b.sy_hash)[base + (w >> 1)];
    }
}

// ---------------------------------------------------------------------------
// index access (StrobemerIndex, step2/index.hpp:57-147)

__device__ __forceinline__ uint64_t rec_hash(const DevIndex &ix, uint64_t x) {
    return reinterpret_cast<const uint64_t *>(ix.rs)[2 * x];
}

// first index of the bucket range holding key, or GIS_NOT_FOUND
// (StrobemerIndex::find, step2/index.hpp:57-81: linear scan of a small bucket,
// lower_bound otherwise; both return the first equal entry). *scan is the
// record count of the byte model: the records a linear scan reads up to the
// first hash >= key (all of them when there is none), whichever search ran.
__device__ __forceinline__ uint64_t dev_find_in(const DevIndex &ix, uint64_t key, uint64_t s, uint64_t e,
                                               uint32_t *scan) {
    uint32_t pr = 0;
    uint64_t res = GIS_NOT_FOUND;
    if (s == e) {
    } else if (e - s < 8) {
        for (uint64_t x = s; x < e; x++) {
            const uint64_t h = rec_hash(ix, x);
            pr++;
            if (h >= key) {
                res = h == key ? x : GIS_NOT_FOUND;
                break;
            }
        }
    } else {
        uint64_t lo = s, cnt = e - s;
        while (cnt > 0) {
            const uint64_t step = cnt >> 1, it = lo + step;
            pr++;
            if (rec_hash(ix, it) < key) { lo = it + 1; cnt -= step + 1; }
            else cnt = step;
        }
        if (lo < e && rec_hash(ix, lo) == key) res = lo;
        pr = (uint32_t)(lo - s) + (lo < e ? 1u : 0u);
    }
    *scan = pr;
    return res;
}

__device__ __forceinline__ uint64_t dev_find(const DevIndex &ix, uint64_t key, uint32_t *scan) {
    const uint32_t bk = (uint32_t)(key >> (64 - ix.bits));
    return dev_find_in(ix, key, ix.starts[bk], ix.starts[bk + 1], scan);
}

__device__ __forceinline__ uint64_t dev_find(const DevIndex &ix, uint64_t key) {
    uint32_t pr;
    return dev_find(ix, key, &pr);
}

// is_filtered: hash[pos] == hash[pos + filter_cutoff], past-the-end reads as ~0
// (step2/index.hpp:83-93)
__device__ __forceinline__ bool dev_filtered(const DevIndex &ix, uint64_t pos, uint64_t key) {
    const uint64_t x = pos + ix.filter_cutoff;
    const uint64_t hx = x < ix.n ? rec_hash(ix, x) : UINT64_MAX;
    return hx == key;
}

// get_count: length of the equal-hash run at pos inside its bucket
// (step2/index.hpp:115-147)
__device__ __forceinline__ uint32_t dev_get_count(const DevIndex &ix, uint64_t pos) {
    const uint64_t key = rec_hash(ix, pos);
    const uint32_t bk = (uint32_t)(key >> (64 - ix.bits));
    const uint64_t pe = ix.starts[bk + 1];
    if (pe - pos < 8) {
        uint32_t c = 1;
        for (uint64_t x = pos + 1; x < pe; x++) {
            if (rec_hash(ix, x) == key) c++;
            else break;
        }
        return c;
    }
    uint64_t lo = pos, cnt = pe - pos;
    while (cnt > 0) {
        const uint64_t step = cnt >> 1, it = lo + step;
        if (!(key < rec_hash(ix, it))) { lo = it + 1; cnt -= step + 1; }
        else cnt = step;
    }
    return (uint32_t)(lo - pos);
}

// Walk the equal-hash run at pos (add_to_hits_per_ref, step2/nam.cu:45-62):
// keep entry e iff |query span - ref span| <= the running minimum. Counts the
// kept hits, and writes them when out != nullptr; *run receives the run's
// length.
// AHEAD: records loaded together (the walk waits for each load; the lookup's runs,
// of buckets beyond the line, are short)
template <uint32_t AHEAD = 4>
__device__ __forceinline__ uint32_t walk_run(const DevIndex &ix, uint64_t pos, uint64_t key,
                                             int qs, int qe, uint32_t strand_bit, DevHit *out,
                                             uint32_t *run = nullptr) {
    const int qspan = qe - qs;
    int min_diff = 0x7fffffff;
    uint32_t c = 0, rec = 0;
    bool in = pos < ix.n;
    for (uint64_t x = pos; in; x += AHEAD) {
        uint4 v[AHEAD];
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; u++) v[u] = ix.rs[x + u < ix.n ? x + u : ix.n - 1];
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; u++) {
            in = in && x + u < ix.n && ((uint64_t)v[u].x | ((uint64_t)v[u].y << 32)) == key;
            if (!in) break;
            rec++;
            const int rspan = (int)(v[u].w & 0xffu) + ix.k;
            int d = qspan - rspan;
            d = d < 0 ? -d : d;
            if (d <= min_diff) {
                if (out) {
                    DevHit hh;
                    hh.ref_strand = strand_bit | (v[u].w >> 8);
                    hh.ref_start = (int32_t)v[u].z;
                    hh.ref_end = (int32_t)v[u].z + rspan;
                    hh.query_start = (uint16_t)qs;
                    hh.query_end = (uint16_t)qe;
                    out[c] = hh;
                }
                c++;
                min_diff = d;
            }
        }
    }
    if (run) *run = rec;
    return c;
}

// The same walk by the whole wave, 64 records per step, for the long runs of
// the rescue path (up to hard_cutoff records): the running minimum of
// add_to_hits_per_ref is the minimum of all earlier differences (an entry
// that is not kept does not lower it), so entry e is kept iff its difference
// is at most the exclusive prefix minimum at e. Returns the kept count (the
// same on every lane) and writes the kept hits in run order when out !=
// nullptr. Every lane calls it with the same arguments.
constexpr uint32_t WALK_WAVE_MIN = 32;  // runs longer than this take the wave walk
// kept hits above which pooled_hits gives a seed the wave: a lane's walk is a wait
// for memory every AHEAD records, the wave's one every 64
constexpr uint32_t WALK_LANE_MAX = 8;

__device__ __forceinline__ uint32_t walk_run_wave(const DevIndex &ix, uint64_t pos, uint64_t key, int qs, int qe,
                                                  uint32_t strand_bit, DevHit *out) {
    const uint32_t lane = lane_id();
    const int qspan = qe - qs;
    int carry = 0x7fffffff;
    uint32_t kept = 0;
    // (the next records are loaded while these are looked at)
    uint4 next = ix.rs[pos + lane < ix.n ? pos + lane : ix.n - 1];
    for (uint64_t x0 = pos; x0 < ix.n; x0 += 64) {
        const uint4 v = next;
        const uint64_t x = x0 + lane;
        next = ix.rs[x + 64 < ix.n ? x + 64 : ix.n - 1];
        const bool in = x < ix.n && ((uint64_t)v.x | ((uint64_t)v.y << 32)) == key;
        // equal hashes are contiguous: the run ends at the first other record
        const uint64_t other = ballot(!in);
        const uint32_t len = other ? (uint32_t)__builtin_ctzll(other) : 64u;
        const bool valid = lane < len;
        const int rspan = (int)(v.w & 0xffu) + ix.k;
        int d = qspan - rspan;
        d = d < 0 ? -d : d;
        const int incl = ~wave_incl_max(~(valid ? d : 0x7fffffff));
        int excl = __builtin_amdgcn_update_dpp(0x7fffffff, incl, 0x138, 0xf, 0xf, false);  // wave_shr:1
        excl = carry < excl ? carry : excl;
        const bool keep = valid && d <= excl;
        const uint64_t km = ballot(keep);
        if (out && keep) {
            DevHit hh;
            hh.ref_strand = strand_bit | (v.w >> 8);
            hh.ref_start = (int32_t)v.z;
            hh.ref_end = (int32_t)v.z + rspan;
            hh.query_start = (uint16_t)qs;
            hh.query_end = (uint16_t)qe;
            out[kept + mbcnt(km)] = hh;
        }
        kept += (uint32_t)__popcll(km);
        const int last = (int)readlane_u32((uint32_t)incl, 63);
        carry = last < carry ? last : carry;
        if (len < 64) break;
    }
    return kept;
}

// ---------------------------------------------------------------------------
// Probe of one query randstrobe for the per-stage lookup. The result is the
// reference's (StrobemerIndex::find + is_filtered + the run walk of
// add_to_hits_per_ref), reached with fewer dependent memory steps: the
// bucket's line (DevIndex::lines) holds its bounds and first records, so one
// line fetch serves a bucket of at most PROBE_SMALL records (nearly all of
// them: buckets hold about 2.4 records on average). The first equal record,
// the run length (equal hashes never cross a bucket), the filter test and the
// kept hits then follow from registers. Larger buckets take the reference's
// search and the separate filter probe in the table.

constexpr uint32_t PROBE_SMALL = BUCKET_LINE - 1;  // 7: 99.6% of buckets at 2.4 records per bucket

// a table record as the probe reads it (gis_ref_randstrobe)
struct alignas(16) IdxRec {
    uint64_t hash;
    uint32_t position;
    uint32_t packed;  // ref_index << 8 | strobe2 offset
};

struct Probe {
    uint64_t key, s, e, pos;
    IdxRec r[PROBE_SMALL];  // records s, s + 1, ... of a small bucket
    uint32_t scan;          // records a linear scan reads to the first hash >= key (byte model)
    uint32_t run;           // length of the equal-hash run of a kept seed (byte model)
    uint32_t hc;            // kept hits (0 when absent or filtered)
    uint32_t keep;          // small bucket: bit j = record s + j is a kept hit
    bool found, filtered;
};

__device__ __forceinline__ bool probe_small(const Probe &p) { return p.e - p.s <= PROBE_SMALL; }

// Bucket bounds (StrobemerIndex::find, step2/index.hpp:57-62) and the
// bucket's first PROBE_SMALL records, all from the bucket's line: one cache
// line, independent loads, no dependent second fetch. Records past the
// bucket's size are zeros and never compared. A size of 2^32 - 1 or more is
// clamped in the line; such buckets are large, and large buckets search the
// table between the starts[] bounds.
__device__ __forceinline__ void probe_line(const DevIndex &ix, Probe &p) {
    const uint32_t bk = (uint32_t)(p.key >> (64 - ix.bits));
    const uint4 *line = ix.lines + (uint64_t)bk * BUCKET_LINE;
    const uint4 h = line[0];
    const IdxRec *recs = reinterpret_cast<const IdxRec *>(line + 1);
#pragma unroll
    for (uint32_t j = 0; j < PROBE_SMALL; j++) p.r[j] = recs[j];
    p.s = (uint64_t)h.x | ((uint64_t)h.y << 32);
    p.e = p.s + h.z;
}

// Search, filter and run walk. Small buckets: the reference's linear scan
// stops at the first record >= key, which is record s + (records below key);
// the run is the records equal to key; hash[pos + filter_cutoff] == key
// exactly when the run is longer than filter_cutoff (past the bucket the
// hashes differ, past the table the reference reads ~0).
// the first equal record of a small bucket from the line's records:
// records below the key, records equal to it
__device__ __forceinline__ void probe_small_find(Probe &p, uint32_t &lt, uint32_t &eq) {
    const uint32_t sz = (uint32_t)(p.e - p.s);
    lt = 0;
    eq = 0;
#pragma unroll
    for (uint32_t j = 0; j < PROBE_SMALL; j++) {
        const uint64_t h = p.r[j].hash;
        if (j < sz) {
            lt += h < p.key ? 1u : 0u;
            eq += h == p.key ? 1u : 0u;
        }
    }
    p.scan = lt < sz ? lt + 1 : sz;
    p.found = eq > 0;
    p.pos = p.found ? p.s + lt : GIS_NOT_FOUND;
}

__device__ __forceinline__ void probe_finish(const DevIndex &ix, Probe &p, int qs, int qe) {
    p.hc = 0;
    p.keep = 0;
    p.run = 0;
    p.filtered = false;
    if (probe_small(p)) {
        uint32_t lt, eq;
        probe_small_find(p, lt, eq);
        if (!p.found) return;
        p.filtered = eq > ix.filter_cutoff ||
                     (p.key == UINT64_MAX && p.pos + ix.filter_cutoff >= ix.n);
        const int qspan = qe - qs;
        int min_diff = 0x7fffffff;
#pragma unroll
        for (uint32_t j = 0; j < PROBE_SMALL; j++) {
            if (j >= lt && j < lt + eq) {
                int d = qspan - ((int)(p.r[j].packed & 0xffu) + ix.k);
                d = d < 0 ? -d : d;
                if (d <= min_diff) {
                    p.keep |= 1u << j;
                    p.hc++;
                    min_diff = d;
                }
            }
        }
        // a filtered seed has no hits, but a rescued read may still take its run
        p.hc = p.filtered ? 0u : p.hc;
        p.run = p.filtered ? 0u : eq;
        return;
    }
    p.pos = p.e - p.s < 0xffffffffull ? dev_find_in(ix, p.key, p.s, p.e, &p.scan) : dev_find(ix, p.key, &p.scan);
    p.found = p.pos != GIS_NOT_FOUND;
    if (!p.found) return;
    p.filtered = dev_filtered(ix, p.pos, p.key);
    if (p.filtered) return;
    p.hc = walk_run<1>(ix, p.pos, p.key, qs, qe, 0u, nullptr, &p.run);
}

// the kept hits of a probe, in run order
__device__ __forceinline__ void probe_emit(const DevIndex &ix, const Probe &p, int qs, int qe,
                                           uint32_t strand_bit, DevHit *out) {
    if (!probe_small(p)) {
        walk_run<1>(ix, p.pos, p.key, qs, qe, strand_bit, out);
        return;
    }
    uint32_t c = 0;
#pragma unroll
    for (uint32_t j = 0; j < PROBE_SMALL; j++) {
        if ((p.keep >> j) & 1u) {
            DevHit hh;
            hh.ref_strand = strand_bit | (p.r[j].packed >> 8);
            hh.ref_start = (int32_t)p.r[j].position;
            hh.ref_end = (int32_t)p.r[j].position + (int)(p.r[j].packed & 0xffu) + ix.k;
            hh.query_start = (uint16_t)qs;
            hh.query_end = (uint16_t)qe;
            out[c++] = hh;
        }
    }
}

// ---------------------------------------------------------------------------
// per-stage: lookup + filter + hit count per randstrobe; nonrepetitive
// fraction and the rescue decision per read (find_nams, step2/nam.cu:553-732,
// and the caller's test, step2/main.cu:3209-3216). One randstrobe per lane,
// 64 per pass; a 150 bp read's ~42 randstrobes fill one pass. While the
// read's hits fit its region of the hit array they are written there in seed
// order; a read with more hits takes a place in the pool, and k_hits writes
// them.
//
// Write traffic is part of this kernel's bound, so a one-pass read (at most
// 64 randstrobes) keeps its per-randstrobe results (position, kept-hit count)
// in registers and stores them only when k_hits reads them: when the read is
// rescued or its hits go to the pool. Longer reads, and the fused kernel's spilled reads, store them
// in every pass. Wave sums and scans use DPP (52 VGPRs).
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(6))) void k_lookup(
    DevBatch b, ReadSet set, DevIndex ix, int rescue_mode, int keep_spill) {
    const uint32_t lane = lane_id();
    const uint32_t cnt = set_count(set);
    for (uint32_t w = wave_index(WPB); w < cnt; w += gridDim.x * WPB) {
        const uint32_t r = set.ids ? sload(set.ids + w) : w;
        const uint32_t n = sload(b.rs_cnt + r);
        const uint64_t base = sload(b.rs_off + r);
        const uint32_t half = sload(b.rs_nfwd + r);
        // results stay in registers for a one-pass read the decision below
        // does not hand to a later kernel
        const bool defer = n <= 64 && !keep_spill && rescue_mode != 2;
        uint32_t found = 0, good = 0, hits = 0, bytes = 0, streams = 0;
        uint64_t pos0 = GIS_NOT_FOUND;
        uint32_t hc0 = 0;
        DevHit *region = b.hits + (uint64_t)r * HIT_REGION;
        // the regions must lie inside the hit array (else every read pools)
        const bool region_ok = (uint64_t)(r + 1) * HIT_REGION <= b.hit_cap;
        for (uint32_t i0 = 0; i0 < n; i0 += 64) {
            // straight-line loads (lanes past the end repeat the last item)
            const uint32_t i = i0 + lane;
            const bool act = i < n;
            const uint64_t x = base + (act ? i : n - 1);
            Probe P;
            P.key = b.rs_hash[x];
            const uint32_t span = b.rs_span[x];
            const int qs = (int)span_start(span), qe = (int)span_end(span);
            probe_line(ix, P);
            // the scheduler may not hoist uses of the line between its loads
            __builtin_amdgcn_sched_barrier(0);
            uint32_t by = 0, sb = 0;
            if (act) {
                probe_finish(ix, P, qs, qe);
                // the table bytes of the search: the bucket bounds (16), the
                // records a linear scan reads to the first hash >= key; a
                // found seed's filter probe (8), and a kept one's run past
                // its first record plus the hash that ends it: 16 per run
                // record in all. Beside them the streams: the query in (12)
                // and, where stored, the result out (12).
                by = 16 + 16 * P.scan;
                if (P.found) by += P.filtered ? 8u : 16u * P.run;
                sb = 12;
                if (defer) {
                    pos0 = P.pos;
                    hc0 = P.hc;
                } else {
                    b.pos[base + i] = P.pos;
                    b.hcnt[base + i] = P.hc;
                    sb += 12;
                }
            } else {
                P.hc = 0;
                P.found = false;
                P.filtered = false;
            }
            found += wave_count(act && P.found);
            good += wave_count(act && P.found && !P.filtered);
            const uint32_t incl = wave_incl_scan_dpp(P.hc);
            const uint32_t chunk_hits = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            // while the read's hits fit its region, write them there in seed
            // order: 16 per hit
            if (region_ok && hits + chunk_hits <= HIT_REGION) {
                if (P.hc > 0)
                    probe_emit(ix, P, qs, qe, i >= half ? 0x80000000u : 0u, region + hits + (incl - P.hc));
                sb += 16 * P.hc;
            }
            hits += chunk_hits;
            bytes += wave_sum_dpp(by);
            streams += wave_sum_dpp(sb);
        }
        const float frac = found > 0 ? (float)good / (float)found : 1.0f;
        const bool rescue = rescue_mode == 2 || (rescue_mode == 0 && ((double)frac < 0.7 || hits == 0));
        const bool pooled = !rescue && hits > 0 && (hits > HIT_REGION || !region_ok);
        // (a rescued read none of whose seeds is in the table has no hits either way)
        const bool listed = rescue && found > 0;
        if (defer && (listed || pooled)) {
            if (lane < n) {
                b.pos[base + lane] = pos0;
                b.hcnt[base + lane] = hc0;
            }
            streams += 12 * n;
        }
        if (lane == 0) {
            b.lk_bytes[r] = bytes;
            b.lk_stream[r] = streams;
            b.frac[r] = frac;
            const uint8_t keep = keep_spill ? (uint8_t)(b.flags[r] & FLAG_SPILL) : (uint8_t)0;
            b.flags[r] = (uint8_t)(keep | (rescue ? GIS_FLAG_RESCUED : 0) |
                                   (n == 0 ? GIS_FLAG_NO_RANDSTROBES : 0));
            b.hit_total[r] = rescue ? 0u : hits;  // rescued reads discard these hits
            b.rhit_total[r] = 0;
            b.rhit_off[r] = 0;
            // hits beyond the read's region: a place in the pool, and k_hits
            // writes them
            uint64_t off = (uint64_t)r * HIT_REGION;
            if (pooled) {
                off = (uint64_t)b.n_reads * HIT_REGION + atomicAdd(&b.ctl->hit_pool, (unsigned long long)hits);
                b.sel_ids[2ull * b.n_reads + atomicAdd(&b.ctl->n_sel[SEL_POOLED], 1u)] = r;
            }
            b.hit_off[r] = off;
            // (one counter takes an append every ~7 ns: 12 000 reads too short for
            // any seed, a third of 36 617 of 50 to 101 bp, took 90 us here and 90
            // more in k_hits)
            if (listed) b.sel_ids[atomicAdd(&b.ctl->n_sel[SEL_RESCUED], 1u)] = r;
        }
    }
}

// the hits of a read that did not fit its region, into the pool (same walk as
// k_lookup)
__device__ __forceinline__ void pooled_hits(const DevBatch &b, const DevIndex &ix, uint32_t r) {
    const uint32_t lane = lane_id();
    const uint32_t n = sload(b.rs_cnt + r);
    const uint64_t base = sload(b.rs_off + r);
    const uint32_t half = sload(b.rs_nfwd + r);
    DevHit *out = b.hits + sload(b.hit_off + r);
    uint32_t carry = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
        const uint32_t i = i0 + lane;
        const uint32_t hc = i < n ? b.hcnt[base + i] : 0u;
        const uint32_t incl = wave_incl_scan_dpp(hc);
        if (hc > 0 && hc <= WALK_LANE_MAX)
            walk_run(ix, b.pos[base + i], b.rs_hash[base + i], (int)span_start(b.rs_span[base + i]),
                     (int)span_end(b.rs_span[base + i]), i >= half ? 0x80000000u : 0u, out + carry + incl - hc);
        // long runs: the whole wave walks each one
        for (uint64_t cm = ballot(hc > WALK_LANE_MAX); cm; cm &= cm - 1) {
            const uint32_t l = (uint32_t)__builtin_ctzll(cm), il = i0 + l;
            const uint64_t xl = base + il;
            walk_run_wave(ix, b.pos[xl], b.rs_hash[xl], (int)span_start(b.rs_span[xl]), (int)span_end(b.rs_span[xl]),
                          il >= half ? 0x80000000u : 0u, out + carry + readlane_u32(incl - hc, l));
        }
        carry += readlane_u32(incl, 63);
    }
}

// ---------------------------------------------------------------------------
// rescue (find_nams_rescue, step2/nam.cu:927-984)
//
// A seed is taken when count <= hard_cutoff and (count <= rescue_cutoff or
// fewer than 5 seeds of its strand precede it in (count, query_start,
// query_end) order): exactly the prefix the reference's sorted loop keeps
// (step2/nam.cu:957-972). Taken seeds walk their runs in query_start order,
// which is the seeds' own order within a strand.

__device__ __forceinline__ bool rh_less(uint32_t ca, uint32_t qa, uint32_t ea, uint32_t cb,
                                        uint32_t qb, uint32_t eb) {
    return ca < cb || (ca == cb && (qa < qb || (qa == qb && ea < eb)));
}

// The rescue of one read: counts of its seeds, the taken ones' hits, a place
// for them in rhits (one atomic per read), and the hits. A read whose hits do
// not fit rhits is left out (the host grows it to rhit_pool and runs again).
__device__ __forceinline__ void rescued_hits(const DevBatch &b, const DevIndex &ix, uint32_t r,
                                             uint32_t rescue_cutoff, uint32_t hard_cutoff) {
    const uint32_t lane = lane_id();
    const uint32_t n = sload(b.rs_cnt + r);
    const uint64_t base = sload(b.rs_off + r);
    const uint32_t half = sload(b.rs_nfwd + r);
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
        const uint32_t i = i0 + lane;
        if (i < n) {
            const uint64_t pos = b.pos[base + i];
            b.hcnt[base + i] = pos != GIS_NOT_FOUND ? dev_get_count(ix, pos) : 0u;
        }
    }
    wave_sync_mem();
    uint32_t total = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
        const uint32_t i = i0 + lane;
        uint32_t rh = 0;
        bool coop = false;
        if (i < n) {
            const uint32_t c = b.hcnt[base + i];
            bool taken = false;
            if (c > 0 && c <= hard_cutoff) {
                taken = c <= rescue_cutoff;
                if (!taken) {
                    const uint32_t lo = i < half ? 0 : half, hi = i < half ? half : n;
                    const uint32_t sp = b.rs_span[base + i], qs = span_start(sp), qe = span_end(sp);
                    uint32_t rank = 0;
                    for (uint32_t j = lo; j < hi && rank < 5; j++) {
                        const uint32_t cj = b.hcnt[base + j];
                        if (cj == 0) continue;
                        const uint32_t spj = b.rs_span[base + j];
                        rank += rh_less(cj, span_start(spj), span_end(spj), c, qs, qe) ? 1u : 0u;
                    }
                    taken = rank < 5;
                }
            }
            if (taken && c <= WALK_WAVE_MIN)
                rh = walk_run(ix, b.pos[base + i], b.rs_hash[base + i], (int)span_start(b.rs_span[base + i]),
                              (int)span_end(b.rs_span[base + i]), 0u, nullptr);
            coop = taken && c > WALK_WAVE_MIN;
        }
        // long runs: the whole wave walks each one
        uint64_t cm = ballot(coop);
        while (cm) {
            const uint32_t l = (uint32_t)__builtin_ctzll(cm);
            cm &= cm - 1;
            const uint64_t xl = base + i0 + l;
            const uint32_t k = walk_run_wave(ix, b.pos[xl], b.rs_hash[xl], (int)span_start(b.rs_span[xl]),
                                             (int)span_end(b.rs_span[xl]), 0u, nullptr);
            if (lane == l) rh = k;
        }
        if (i < n) b.rcnt[base + i] = rh;
        total += wave_sum_dpp(rh);
    }
    if (total == 0) return;  // (k_lookup has written that)
    unsigned long long off = 0;
    if (lane == 0) {
        off = atomicAdd(&b.ctl->rhit_pool, (unsigned long long)total);
        b.rhit_total[r] = total;
        b.rhit_off[r] = off;
    }
    off = uni64(off);
    if (off + total > b.rhit_cap) {
        if (lane == 0) atomicOr(&b.ctl->overflow, OVF_RHITS);
        return;
    }
    wave_sync_mem();
    DevHit *out = b.rhits + off;
    uint32_t carry = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
        const uint32_t i = i0 + lane;
        const uint32_t rh = i < n ? b.rcnt[base + i] : 0u;
        // runs longer than WALK_WAVE_MIN take the wave walk, as above
        const bool coop = rh > 0 && b.hcnt[base + i] > WALK_WAVE_MIN;
        const uint32_t incl = wave_incl_scan_dpp(rh);
        if (rh > 0 && !coop)
            walk_run(ix, b.pos[base + i], b.rs_hash[base + i], (int)span_start(b.rs_span[base + i]),
                     (int)span_end(b.rs_span[base + i]), i >= half ? 0x80000000u : 0u, out + carry + incl - rh);
        uint64_t cm = ballot(coop);
        while (cm) {
            const uint32_t l = (uint32_t)__builtin_ctzll(cm);
            cm &= cm - 1;
            const uint32_t il = i0 + l;
            const uint64_t xl = base + il;
            walk_run_wave(ix, b.pos[xl], b.rs_hash[xl], (int)span_start(b.rs_span[xl]), (int)span_end(b.rs_span[xl]),
                          il >= half ? 0x80000000u : 0u, out + carry + readlane_u32(incl - rh, l));
        }
        carry += readlane_u32(incl, 63);
    }
}

// the reads that k_lookup listed, one per wave: pooled ones, then rescued ones
__global__ __launch_bounds__(64 * WPB) void k_hits(DevBatch b, DevIndex ix, uint32_t rescue_cutoff,
                                                   uint32_t hard_cutoff) {
    const uint32_t n_pool = sload(&b.ctl->n_sel[SEL_POOLED]), n_resc = sload(&b.ctl->n_sel[SEL_RESCUED]);
    const bool pool_ok = (uint64_t)b.n_reads * HIT_REGION + sload(&b.ctl->hit_pool) <= b.hit_cap;
    if (n_pool && !pool_ok && blockIdx.x == 0 && threadIdx.x == 0) atomicOr(&b.ctl->overflow, OVF_HITS);
    for (uint32_t w = wave_index(WPB); w < n_pool + n_resc; w += gridDim.x * WPB) {
        if (w >= n_pool)
            rescued_hits(b, ix, uni32(b.sel_ids[w - n_pool]), rescue_cutoff, hard_cutoff);
        else if (pool_ok)
            pooled_hits(b, ix, uni32(b.sel_ids[2ull * b.n_reads + w]));
        wave_sync_mem();
    }
}

// a hit array overflowed (an earlier kernel found it): the host grows it and
// runs again, and the kernels after the hits leave their work out
__device__ __forceinline__ bool hits_missing(const DevBatch &b) {
    return (sload(&b.ctl->overflow) & (OVF_HITS | OVF_RHITS)) != 0;
}

// ---------------------------------------------------------------------------
// NAM merge (merge_hits_into_nams, step2/nam.cu:347-513). Hits of a read
// arrive strand by strand, seeds in query_start order and each run in table
// order; within one (strand, ref) group that is (query_start, ref_start)
// order, the order the reference sorts each group into (step2/nam.cu:373).
// The hits are grouped by (strand, ref_id) with a stable sort and each group
// is merged in that order: every hit extends or is contained in the first
// open NAM (in creation order) that accepts it, or opens a new NAM
// (step2/nam.cu:391-447). A NAM whose query_end lies before the current
// query_start can never accept a hit again; when it leaves the open list does
// not change any field. Creation order inside a group is canonical order, so
// NAM c of a group is written at (NAMs of earlier groups) + c with nam_id =
// that rank.
//
// The open NAMs of the current group live one per lane; the hit is broadcast
// and a ballot picks the first accepting lane. When 64 lanes are open and
// none can be retired, the group continues on a NAM list in global scratch
// scanned 64 entries at a time (the "wide" form), retiring dead NAMs as the
// list grows.

__device__ __forceinline__ void bitonic_mem(uint64_t *keys, uint32_t P) {
    const uint32_t lane = lane_id();
    for (uint32_t size = 2; size <= P; size <<= 1) {
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            for (uint32_t t0 = 0; t0 < P / 2; t0 += 64) {
                const uint32_t t = t0 + lane;
                if (t < P / 2) {
                    const uint32_t i = (t / stride) * 2 * stride + (t % stride);
                    const uint32_t j = i + stride;
                    const bool asc = (i & size) == 0;
                    const uint64_t a = keys[i], c = keys[j];
                    if ((a > c) == asc) { keys[i] = c; keys[j] = a; }
                }
            }
            wave_sync_mem();
        }
    }
}

constexpr uint32_t MERGE_OVERFLOW = 0xffffffffu;

struct LaneNam {
    int qs, qe, qp, rs, re, rp, n;
    uint32_t cid;
};

__device__ __forceinline__ void lane_nam_store(gis_nam *out, uint32_t idx, uint32_t rsd,
                                               const LaneNam &o) {
    gis_nam x;
    x.nam_id = (int32_t)idx;
    x.query_start = o.qs;
    x.query_end = o.qe;
    x.query_prev_hit_startpos = o.qp;
    x.ref_start = o.rs;
    x.ref_end = o.re;
    x.ref_prev_hit_startpos = o.rp;
    x.n_hits = o.n;
    x.ref_id = (int32_t)(rsd & 0x7fffffffu);
    x.score = nam_score(o.qs, o.qe, o.rs, o.re, o.n);
    x.is_rc = (uint8_t)(rsd >> 31);
    x.pad_[0] = x.pad_[1] = x.pad_[2] = 0;
    out[idx] = x;
}

__device__ __forceinline__ LaneNam from_wide(const WideNam &w) {
    return LaneNam{w.qs, w.qe, w.qp, w.rs, w.re, w.rp, (int)w.n, w.cid};
}

__device__ __forceinline__ int permute_push(int v, uint32_t dst) {
    return __builtin_amdgcn_ds_permute((int)(dst << 2), v);
}

// does open NAM o accept hit (qs, qe, rs, re), and does the hit extend it
__device__ __forceinline__ bool nam_accepts(int o_qp, int o_qe, int o_rp, int o_re, int qs, int qe,
                                            int rs, int re, bool &ext) {
    // bitwise on purpose: no short-circuit branches in the merge loops
    const bool near = (o_qp < qs) & (qs <= o_qe) & (o_rp < rs) & (rs <= o_re);
    ext = (qe > o_qe) & (re > o_re);
    const bool con = (qe <= o_qe) & (re <= o_re);
    return near & (ext | con);
}

// The wide list of one merge: entries below near_cap in `near` (LDS when the
// caller has it), the rest at the same indices of `far`. near_cap is a
// multiple of 64, so the 64 entries of a chunk are all on one side.
// The LDS part is typed as LDS so that its accesses compile to LDS
// instructions rather than flat ones.
typedef __attribute__((address_space(3))) WideNam LdsWideNam;

struct WideList {
    LdsWideNam *near;
    WideNam *far;
    uint32_t near_cap;
};

__device__ __forceinline__ WideNam wget(const WideList &L, uint32_t e) {
    WideNam w;
    if (e < L.near_cap) {
        const LdsWideNam &x = L.near[e];
        w = WideNam{x.qs, x.qe, x.qp, x.rs, x.re, x.rp, x.n, x.cid};
    } else {
        w = L.far[e];
    }
    return w;
}

__device__ __forceinline__ void wput(const WideList &L, uint32_t e, const WideNam &w) {
    if (e < L.near_cap) {
        LdsWideNam &x = L.near[e];
        x.qs = w.qs;
        x.qe = w.qe;
        x.qp = w.qp;
        x.rs = w.rs;
        x.re = w.re;
        x.rp = w.rp;
        x.n = w.n;
        x.cid = w.cid;
    } else {
        L.far[e] = w;
    }
}

// write the wide list's NAMs of the group that ends (all of them are final)
__device__ __forceinline__ void wide_flush(const WideList &wide, uint32_t nw, gis_nam *out, uint32_t base,
                                           uint32_t grp, uint32_t cap) {
    for (uint32_t c0 = 0; c0 < nw; c0 += 64) {
        const uint32_t e = c0 + lane_id();
        if (e < nw) {
            const WideNam w = wget(wide, e);
            if (base + w.cid < cap) lane_nam_store(out, base + w.cid, grp, from_wide(w));
        }
    }
}

// items loaded ahead per lane by the passes over a read's hits: a lone wave's
// time in them is the latency of its loads
constexpr uint32_t AHEAD = 8;

// f(i, item i) for the n items of a read that load gives, AHEAD chunks of 64 at a
// time; lanes beyond the end get the last item, with i >= n
template <typename T, typename Load, typename F>
__device__ __forceinline__ void each_ahead(uint32_t n, Load load, F f) {
    for (uint32_t i0 = 0; i0 < n; i0 += 64 * AHEAD) {
        T v[AHEAD];
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; u++) {
            const uint32_t i = i0 + 64 * u + lane_id();
            v[u] = load(i < n ? i : n - 1);
        }
#pragma unroll
        for (uint32_t u = 0; u < AHEAD; u++) f(i0 + 64 * u + lane_id(), v[u]);
    }
}

// counts to exclusive prefixes over 256 bins, four a lane
__device__ __forceinline__ void bins_prefix(uint32_t *bins) {
    const uint32_t lane = lane_id();
    wave_sync();
    const uint32_t b0 = bins[4 * lane], b1 = bins[4 * lane + 1], b2 = bins[4 * lane + 2], b3 = bins[4 * lane + 3];
    const uint32_t t = b0 + b1 + b2 + b3, at = wave_incl_scan_dpp(t) - t;
    wave_sync();
    bins[4 * lane] = at;
    bins[4 * lane + 1] = at + b0;
    bins[4 * lane + 2] = at + b0 + b1;
    bins[4 * lane + 3] = at + b0 + b1 + b2;
    wave_sync();
}

// The n keys (group << 32 | hit index) that load gives to dst, stable by the digit
// that digit(key) gives; bins: the digits' places, afterwards their ends.
template <typename Load, typename Digit>
__device__ __forceinline__ void radix_scatter(uint32_t n, Load load, Digit digit, uint64_t *dst, uint32_t *bins) {
    each_ahead<uint64_t>(n, load, [&](uint32_t i, uint64_t k) {
        const bool in = i < n;
        const uint32_t d = digit(k);
        // the lanes of the same digit, a ballot a bit (digit by digit took a trip
        // to LDS for each of up to 48 groups)
        uint64_t peers = ballot(in);
#pragma unroll
        for (uint32_t bit = 0; bit < 8; bit++) {
            const uint64_t m = ballot((d >> bit) & 1u);
            peers &= (d >> bit) & 1u ? m : ~m;
        }
        const uint32_t rank = mbcnt(peers);
        uint32_t pos = 0;
        if (in) pos = bins[d] + rank;
        wave_sync();
        if (in && rank == 0) bins[d] = pos + (uint32_t)__popcll(peers);
        wave_sync();
        if (in) dst[pos] = k;
    });
    wave_sync_mem();
}

// Grouped order of nh hits: nullptr when they already are in (strand, ref)
// order, else keys (bitonic in keys, nh <= MERGE_LDS and no keys_alt) or one of
// keys / keys_alt (stable radix sort) holding group << 32 | hit index. bins: 256
// words of LDS (the bitonic sort's keys may lie there). binned: the groups are
// the bins, which hold their ends in the order.
//
// A wave's time here is that of its passes over the hits. The first counts the
// groups of a read on references below 128 as it looks for the largest one, so
// that those need one more, the scatter; others sort compact group keys by 8 bits
// a pass. (A read of 5810 hits alone kept k_merge at 119 us; now 76.)
__device__ __forceinline__ const uint64_t *group_order(uint32_t nh, const DevHit *hits, uint64_t *keys,
                                                      uint64_t *keys_alt, uint32_t *bins, bool &binned) {
    const uint32_t lane = lane_id();
    const uint4 *hv = reinterpret_cast<const uint4 *>(hits);
    for (uint32_t u = lane; u < 256; u += 64) bins[u] = 0;
    wave_sync();
    uint32_t max_ref = 0, last = 0;
    bool unsorted = false;
    each_ahead<uint32_t>(nh, [&](uint32_t i) { return hv[i].x; }, [&](uint32_t i, uint32_t rsd) {
        const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp((int)last, (int)rsd, 0x138, 0xf, 0xf, false);
        last = readlane_u32(rsd, 63);
        max_ref = max(max_ref, rsd & 0x7fffffffu);
        unsorted |= before > rsd;
        if (i < nh) atomicAdd(&bins[rsd >> 31 << 7 | (rsd & 127u)], 1u);
    });
    const uint32_t mr = wave_max_dpp(max_ref);
    binned = mr < 128;
    if (ballot(unsorted) == 0) {
        bins_prefix(bins);  // each bin's start: its end is the next one's
        uint32_t e[4];
        for (uint32_t u = 0; u < 4; u++) e[u] = 4 * lane + u < 255 ? bins[4 * lane + u + 1] : nh;
        wave_sync();
        for (uint32_t u = 0; u < 4; u++) bins[4 * lane + u] = e[u];
        wave_sync();
        return nullptr;
    }
    if (nh <= (uint32_t)MERGE_LDS && !keys_alt) {
        uint32_t P = 1;
        while (P < nh) P <<= 1;
        wave_sync();
        for (uint32_t i = lane; i < P; i += 64) keys[i] = i < nh ? (((uint64_t)hv[i].x << 32) | i) : UINT64_MAX;
        wave_sync_mem();
        bitonic_mem(keys, P);
        binned = false;
        return keys;
    }
    if (binned) {
        bins_prefix(bins);
        radix_scatter(nh, [&](uint32_t i) {
            const uint32_t x = hv[i].x;
            return (uint64_t)(x >> 31 << 7 | x) << 32 | i;
        }, [](uint64_t k) { return (uint32_t)(k >> 32) & 255u; }, keys, bins);
        return keys;
    }
    // compact group key: strand above the bits of the largest ref_id; the first
    // pass makes it from the hits
    const uint32_t rbits = 32u - (uint32_t)__builtin_clz(mr);
    const uint64_t *src = nullptr;
    uint64_t *dst = keys;
    for (uint32_t shift = 0; shift < rbits + 1; shift += 8) {
        auto load = [&](uint32_t i) {
            if (src) return src[i];
            const uint32_t x = hv[i].x;
            return (((uint64_t)(x >> 31) << rbits | (x & 0x7fffffffu)) << 32) | i;
        };
        auto digit = [&](uint64_t k) { return (uint32_t)(k >> (32 + shift)) & 255u; };
        for (uint32_t u = lane; u < 256; u += 64) bins[u] = 0;
        wave_sync();
        each_ahead<uint64_t>(nh, load, [&](uint32_t i, uint64_t k) {
            if (i < nh) atomicAdd(&bins[digit(k)], 1u);
        });
        bins_prefix(bins);
        radix_scatter(nh, load, digit, dst, bins);
        src = dst;
        dst = dst == keys ? keys_alt : keys;
    }
    return src;
}

// Reference-interval bounds of one 64-entry chunk of the wide list: every
// entry's previous hit start is at least lo and its ref end at most hi. Starts only grow and ends are raised with the entry, so the bounds
// stay valid (if loose) until the list is compacted and they are recomputed.
struct ChunkBox {
    int lo, hi;
};

// bounds of the wide list's chunks c0 .. (all of them when c0 == 0)
__device__ __forceinline__ void boxes_rebuild(const WideList &wide, uint32_t nw, ChunkBox *box) {
    for (uint32_t c = 0; c * 64 < nw; c++) {
        const uint32_t e = c * 64 + lane_id();
        int lo = 0x7fffffff, hi = (int)0x80000000;
        if (e < nw) {
            const WideNam w = wget(wide, e);
            lo = w.rp;
            hi = w.re;
        }
        lo = wave_imin(lo);
        hi = wave_imax(hi);
        if (lane_id() == 0) box[c] = ChunkBox{lo, hi};
    }
}

// the NAM list of a strand or group in the lanes of a wave: dead NAMs (query end
// before qs: they can take no further hit) leave, the others move up in order.
// Returns the open count; dst of a dead NAM is out[base + cid].
__device__ __forceinline__ uint32_t retire_lanes(LaneNam &o, int qs, gis_nam *out, uint32_t base, uint32_t grp,
                                                 uint32_t cap) {
    const bool keep = o.qe >= qs;
    const uint64_t km = ballot(keep);
    const uint32_t nk = (uint32_t)__popcll(km);
    if (nk == 64) return nk;
    if (!keep && base + o.cid < cap) lane_nam_store(out, base + o.cid, grp, o);
    const uint32_t dst = keep ? mbcnt(km) : nk + mbcnt(~km);
    o.qs = permute_push(o.qs, dst);
    o.qe = permute_push(o.qe, dst);
    o.qp = permute_push(o.qp, dst);
    o.rs = permute_push(o.rs, dst);
    o.re = permute_push(o.re, dst);
    o.rp = permute_push(o.rp, dst);
    o.n = permute_push(o.n, dst);
    o.cid = (uint32_t)permute_push((int)o.cid, dst);
    return nk;
}

// One hit against the NAMs of a wave's lanes: the first of the accepting lanes acc
// takes it, else the lane `free` (its one bit; lanes from there on accept
// nothing) opens a NAM with it. Returns the lane's bit, 0 when no lane can: then
// nothing changed. mk: that bit if it opened one. Masks and selects, no
// branches: the hit and the masks live in scalar registers.
__device__ __forceinline__ uint64_t lanes_take(LaneNam &o, uint64_t acc, uint64_t ext, uint64_t free, uint64_t &mk,
                                               uint32_t cid, int qs, int qe, int rs, int re) {
    const uint64_t x = acc | free, me = x & (0 - x);
    mk = me & free;
    const bool b_me = lane_bit(me), b_mk = lane_bit(mk), b_end = lane_bit(mk | (me & ext));
    o.qs = b_mk ? qs : o.qs;
    o.rs = b_mk ? rs : o.rs;
    o.cid = b_mk ? cid : o.cid;
    o.qe = b_end ? qe : o.qe;
    o.re = b_end ? re : o.re;
    o.qp = b_me ? qs : o.qp;
    o.rp = b_me ? rs : o.rp;
    o.n += b_me ? 1 : 0;  // (0 on a free lane)
    return me;
}

// The hits after hit t of the 64 in a wave's lanes (c, m of them) that the NAM on
// lane w, which took hit t, takes one after the other: with no live NAM of its
// group on a lower lane it is the first to accept each of them as long as it does.
// A hit of the run sees the one before it as the previous hit and the ends' maxima
// so far as the NAM's ends (a hit raises both or neither), so one prefix maximum
// tests the 64 at once. Returns the last hit taken (t if none is).
__device__ __forceinline__ uint32_t take_run(LaneNam &o, uint32_t w, const uint4 &c, uint32_t t, uint32_t m) {
    const uint32_t lane = lane_id();
    const int qs = (int)(c.w & 0xffffu), rs = (int)c.y;
    const uint64_t after = ~0ull << t;  // t and the hits after it
    const uint64_t from = after & (after - 1);
    const bool in = lane_bit(from);
    const int qe_t = __builtin_amdgcn_readlane(o.qe, (int)w), re_t = __builtin_amdgcn_readlane(o.re, (int)w);
    const int qe = in ? (int)(c.w >> 16) : qe_t, re = in ? (int)c.z : re_t;
    const int hq = wave_incl_max(qe), hr = wave_incl_max(re);
    auto before = [](int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, false); };  // wave_shr:1
    const int pq = before(hq), pr = before(hr);
    const uint64_t ok = ballot((uint32_t)before((int)c.x) == c.x) & ballot(before(qs) < qs) & ballot(qs <= pq) &
                        ballot(before(rs) < rs) & ballot(rs <= pr) & ~(ballot(qe > pq) ^ ballot(re > pr));
    const uint64_t stop = (~ok & from) | (m < 64 ? ~0ull << m : 0ull);
    const uint32_t last = (stop ? (uint32_t)__builtin_ctzll(stop) : 64u) - 1;
    const bool me = lane == w;
    o.qe = me ? __builtin_amdgcn_readlane(hq, (int)last) : o.qe;
    o.re = me ? __builtin_amdgcn_readlane(hr, (int)last) : o.re;
    o.qp = me ? __builtin_amdgcn_readlane(qs, (int)last) : o.qp;
    o.rp = me ? __builtin_amdgcn_readlane(rs, (int)last) : o.rp;
    o.n += me ? (int)(last - t) : 0;
    return last;
}

constexpr uint32_t ARRIVAL_BLOCK = 4;
// a strand of more groups than this and more NAMs than lanes is merge_range's (reads
// in repeats)
constexpr uint32_t ARRIVAL_GROUPS = 8;

// Merge of a read's hits in arrival order on one wave, a NAM a lane, without
// grouping them: NAMs of every group of the current strand share the lanes, and
// a NAM only accepts hits of its own group, which arrive in (query_start,
// ref_start) order. A strand's NAMs are ranked by (ref_id, creation) when its
// hits end. With one group on the strand (a read of one place, the usual case)
// creation order is the rank, so dead NAMs may leave when the lanes are full. With
// more, a strand that fills the lanes goes again, one group after the other.
// Returns the NAM count (entries at index >= cap are not written), or
// MERGE_OVERFLOW when a group needs more than 64 lanes (or such a strand has more
// than ARRIVAL_GROUPS groups), or, with BLOCKS, when the hits come in blocks of ARRIVAL_BLOCK or more equal query starts on
// average (repeats): merge_range takes a block at a time.
//
// A lone wave's time is its chain of instructions a hit (one issues every ~8
// cycles), branches above all: the loop over hits has none but its end, the
// full-lanes exit and the run's (~550 cycles a hit; the group-by-group merge took
// ~800 with its sort and block tests before it). Most hits come in runs that one
// NAM takes (of a long read's 128 hits, 78 in two runs, take_run). 8191 reads of
// 400 to 2500 bp, 4230 of them here: k_merge 240 us before, 196 with the runs
// (then the time of three reads with more NAMs than lanes on several references,
// which went to merge_range), 74 with those taken group by group.
template <bool BLOCKS = false>
__device__ __forceinline__ uint32_t merge_arrival(const DevHit *hits, uint32_t nh, gis_nam *out, uint32_t cap) {
    const uint32_t lane = lane_id();
    const uint4 *hv = reinterpret_cast<const uint4 *>(hits);
    // forward hits, and whether a strand holds more than one group (against its
    // first forward and its last reverse hit)
    uint32_t nf = 0;
    bool other[2] = {false, false};
    {
        const uint32_t h0 = uni32(hv[0].x), hl = uni32(hv[nh ? nh - 1 : 0].x);
        uint64_t of = 0, orv = 0;
        uint32_t blocks = 0;
        for (uint32_t y0 = 0; y0 < nh; y0 += 256) {
            // (four loads in flight: a lone wave waits for each)
            uint32_t r4[4], w4[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; u++) {
                const uint32_t x = y0 + 64 * u + lane;
                r4[u] = x < nh ? hv[x].x : 0xffffffffu;
                w4[u] = BLOCKS && x < nh ? hv[x].w & 0xffffu : 0u;
            }
#pragma unroll
            for (uint32_t u = 0; u < 4; u++) {
                const uint32_t x0 = y0 + 64 * u;
                if (x0 >= nh) break;
                const bool in = x0 + lane < nh;
                if (BLOCKS) {
                    const uint32_t pq = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w4[u], 0x138, 0xf, 0xf, false);
                    blocks += wave_count(in && (lane == 0 || w4[u] != pq));
                }
                const uint64_t fwd = ballot(r4[u] >> 31 == 0);
                nf += (uint32_t)__popcll(fwd);
                of |= ballot(r4[u] != h0) & fwd;
                orv |= ballot(in && r4[u] != hl) & ~fwd;
            }
        }
        other[0] = of != 0;
        other[1] = orv != 0;
        if (BLOCKS && nh >= ARRIVAL_BLOCK * blocks) return MERGE_OVERFLOW;
    }
    uint32_t base = 0;
    for (int strand = 0; strand < 2; strand++) {
        const uint32_t xb = strand ? nf : 0u, xe = strand ? nh : nf;
        bool multi = other[strand];
        // the group whose hits alone are taken (`each`), and how many there were
        bool each = false;
        uint32_t grp = 0, n_grp = 0;
        for (;;) {
            LaneNam o{0, 0, 0, 0, 0, 0, 0, 0};
            uint32_t rsd_o = 0xffffffffu;  // this lane's group (no hit's when the lane is free)
            uint32_t made = 0;
            uint64_t free = 1;
            uint32_t after = 0xffffffffu;  // the least group above grp
            bool full = false;
            uint4 next = make_uint4(0u, 0u, 0u, 0u);
            if (xb + lane < xe) next = hv[xb + lane];
            for (uint32_t x0 = xb; x0 < xe && !full; x0 += 64) {
                const uint4 c = next;
                if (x0 + 64 + lane < xe) next = hv[x0 + 64 + lane];
                const uint32_t m = xe - x0 < 64 ? xe - x0 : 64;
                uint64_t todo = ~0ull >> (64 - m);
                if (each) {
                    if (lane < m && c.x > grp) after = min(after, c.x);
                    todo &= ballot(c.x == grp);
                }
                while (todo) {
                    uint32_t rsd = 0;
                    int qs = 0;
                    uint64_t me;
                    do {
                        const uint32_t t = (uint32_t)__builtin_ctzll(todo);
                        rsd = readlane_u32(c.x, t);
                        const uint32_t q = readlane_u32(c.w, t);
                        const int rs = (int)readlane_u32(c.y, t), re = (int)readlane_u32(c.z, t), qe = (int)(q >> 16);
                        qs = (int)(q & 0xffffu);
                        const uint64_t xq = ballot(qe > o.qe), xr = ballot(re > o.re);
                        const uint64_t live = ballot(rsd_o == rsd) & ballot(qs <= o.qe);
                        const uint64_t acc =
                            live & ballot(o.qp < qs) & ballot(o.rp < rs) & ballot(rs <= o.re) & ~(xq ^ xr);
                        uint64_t mk;
                        me = lanes_take(o, acc, xq & xr, free, mk, made, qs, qe, rs, re);
                        rsd_o = lane_bit(mk) ? rsd : rsd_o;
                        const uint32_t fresh = mk != 0 ? 1u : 0u;
                        made += fresh;
                        free <<= fresh;
                        if (me == 0) break;  // no room: the hit waits
                        todo &= todo - 1;
                        // taken by the first live NAM
                        if (me == (live & (0 - live)))
                            todo &= ~0ull << 1 << take_run(o, (uint32_t)__builtin_ctzll(me), c, t, m);
                    } while (todo);
                    if (me != 0) break;
                    if (multi) {
                        // (its groups so far)
                        uint64_t nams = ~0ull;
                        uint32_t k = 0;
                        for (; nams && k <= ARRIVAL_GROUPS; k++)
                            nams &= ~ballot(rsd_o == readlane_u32(rsd_o, (uint32_t)__builtin_ctzll(nams)));
                        if (k > ARRIVAL_GROUPS) return MERGE_OVERFLOW;
                        full = true;
                        break;
                    }
                    const uint32_t n_open = retire_lanes(o, qs, out, base, rsd, cap);
                    if (n_open == 64) return MERGE_OVERFLOW;
                    rsd_o = lane < n_open ? rsd_o : 0xffffffffu;
                    o.n = lane < n_open ? o.n : 0;
                    free = 1ull << n_open;
                }
            }
            if (full) {
                // more NAMs than lanes, of several groups: the groups one by one
                // (nothing of the strand is written yet), least one first
                uint32_t least = 0xffffffffu;
                for (uint32_t x = xb + lane; x < xe; x += 64) least = min(least, hv[x].x);
                multi = false;
                each = true;
                grp = wave_umin(least);
                n_grp = 1;
                continue;
            }
            // the NAMs are final
            uint32_t rank = o.cid;
            if (multi) {  // nothing was retired: NAM c sits on lane c
                rank = 0;
                for (uint32_t q = 0; q < made; q++) {
                    const uint32_t k = readlane_u32(rsd_o, q);
                    rank += (k < rsd_o) | ((k == rsd_o) & (q < lane)) ? 1u : 0u;
                }
            }
            if (o.n > 0 && base + rank < cap) lane_nam_store(out, base + rank, rsd_o, o);
            base += made;
            if (!each) break;
            grp = wave_umin(after);
            if (grp == 0xffffffffu) break;
            if (++n_grp > ARRIVAL_GROUPS) return MERGE_OVERFLOW;
        }
    }
    return base;
}

// LDS of one wave's block matching: the 64 hits in its registers (ref start, ref
// end, query end), and who holds them
struct alignas(16) BlockLds {
    int4 h[64];
    uint32_t hold[64];
};

// The hits that the lanes' NAMs (those of `can`) take of a block: hits [t, t +
// len) of B, ref starts ascending, less those not in cm. Hit by hit, each takes
// the first accepting NAM that no earlier hit of the block took. All hits rank
// the NAMs alike (by lane) and all NAMs the hits (by order), so that assignment
// is also the one where each NAM, in lane order, takes the first accepting hit
// that is left, and the only stable one: NAMs propose to their first accepting
// hit, a hit holds its lowest lane, and a NAM that is turned down goes on to its
// next. A NAM's candidates are the hits with ref start in (o_rp, o_re], found by
// binary search. Returns this lane's hit or -1; took: the hits taken.
//
// A tandem repeat's block has hundreds of hits and NAMs, each NAM with a handful
// of candidates. The hit-by-hit loop took ~25 instructions a hit for every chunk
// of NAMs; this is ~150 for a chunk and 64 hits, most of them waiting for LDS,
// so the candidates are read four at a time.
__device__ __forceinline__ int match_block(BlockLds &B, uint32_t t, uint32_t len, uint64_t cm, bool can, int o_qe,
                                           int o_rp, int o_re, uint64_t &took) {
    const uint32_t lane = lane_id(), end = t + len;
    uint32_t i = t, n = len;  // the first hit with ref start above o_rp
    while (n > 0) {
        const uint32_t half = n >> 1;
        const bool up = B.h[i + half].x <= o_rp;
        i = up ? i + half + 1 : i;
        n = up ? n - half - 1 : half;
    }
    uint64_t mask = 0;
    bool more = can && i < end;
    while (ballot(more)) {
        int4 h[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) h[u] = B.h[min(i + u, end - 1)];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            more = more && i < end && h[u].x <= o_re;
            if (more && ((h[u].z > o_qe) == (h[u].y > o_re))) mask |= 1ull << i;
            i++;
        }
        more = more && i < end;
    }
    mask &= cm;
    B.hold[lane] = 0xffffffffu;
    wave_sync();
    int p;
    for (;;) {
        p = mask ? (int)__builtin_ctzll(mask) : -1;
        if (p >= 0) atomicMin(&B.hold[p], lane);
        wave_sync();
        const bool down = p >= 0 && B.hold[p] != lane;
        if (ballot(down) == 0) break;
        if (down) mask &= mask - 1;
        wave_sync();
    }
    took = ballot(B.hold[lane] != 0xffffffffu);
    wave_sync();
    return p;
}

// blocks of fewer hits go hit by hit
constexpr uint32_t MATCH_MIN = 8;

// Merge hits order[xb .. xe) (hit indices in grouped order; order nullptr:
// the hits themselves in order). NAM c of the k-th group of the range is
// written at out[(NAMs of the range's earlier groups) + c]; entries at index
// >= cap are not written. Returns the NAM count, or MERGE_OVERFLOW when a group
// needs more than 64 open NAMs and there is no wide list.
// box (may be nullptr): bounds of up to box_cap chunks of the wide list. A
// hit can only be accepted by an entry with previous hit start < ref start <=
// ref end, so the scan for the first accepting entry visits only the chunks
// whose bounds admit the hit, in order: the same entry as a full scan.
//
// The hits go block by block: hits of one group and query start. No NAM can take
// two of a block (a NAM that takes one gets previous start qs, and so does one
// that a hit of the block opens), so each meets the NAMs as they were before
// the block. Their acceptance masks are independent; only the assignment, in
// hit order (the first accepting NAM that no earlier hit of the block took,
// else a new one), runs hit by hit, on scalars. A block cut by the end of the
// 64 hits in registers is two blocks.
__device__ __forceinline__ uint32_t merge_range(const DevHit *hits, const uint64_t *order, uint32_t xb,
                                                uint32_t xe, const WideList wide, gis_nam *out,
                                                uint32_t cap, BlockLds &B, ChunkBox *box = nullptr,
                                                uint32_t box_cap = 0) {
    const uint32_t lane = lane_id();
    LaneNam o{0, 0, 0, 0, 0, 0, 0, 0};
    uint32_t n_open = 0, grp = 0xffffffffu, base = 0, gcnt = 0;
    bool wide_mode = false;
    uint32_t nw = 0, wide_mark = 0;
    // the next 64 hits load while these merge (their place in the grouped order
    // was read one step before)
    const uint4 *hv = reinterpret_cast<const uint4 *>(hits);
    const auto place = [&](uint32_t x) {
        const uint32_t i = min(x + lane, xe - 1);
        return order ? (uint32_t)order[i] : i;
    };
    uint32_t at_next = 0;
    uint4 h_next = make_uint4(0u, 0u, 0u, 0u);
    if (xb < xe) {
        h_next = hv[place(xb)];
        at_next = place(xb + 64);
    }
    for (uint32_t x0 = xb; x0 < xe; x0 += 64) {
        const uint4 h = h_next;
        if (x0 + 64 < xe) {
            h_next = hv[at_next];
            at_next = place(x0 + 128);
        }
        const uint32_t c_rsd = h.x, c_rs = h.y, c_re = h.z, c_q = h.w;
        const uint32_t m = xe - x0 < 64 ? xe - x0 : 64;
        // lanes that start a block, and a group (lane 0 against the last chunk's)
        const uint32_t p_rsd = (uint32_t)__shfl_up((int)c_rsd, 1, 64), p_q = (uint32_t)__shfl_up((int)c_q, 1, 64);
        const uint64_t gheads = ballot(c_rsd != (lane ? p_rsd : grp));
        const uint64_t heads = gheads | ballot(((c_q ^ p_q) & 0xffffu) != 0 || lane == 0);
        // hits whose ref start lies below the one before them in their block (a
        // block of one seed has none)
        const int p_rs = __shfl_up((int)c_rs, 1, 64);
        const uint64_t falls = ballot((int)c_rs < p_rs) & ~heads;
        wave_sync();
        B.h[lane] = make_int4((int)c_rs, (int)c_re, (int)(c_q >> 16), 0);
        wave_sync();
        uint32_t singles_until = 0;  // the rest of a block that did not fit the lanes goes hit by hit
        for (uint32_t t = 0; t < m;) {
            const uint32_t q = readlane_u32(c_q, t);
            const int qs = (int)(q & 0xffffu);
            const uint64_t next = heads & ~((2ull << t) - 1);
            const uint32_t len = (next ? min((uint32_t)__builtin_ctzll(next), m) : m) - t;
            const uint64_t block = (len >= 64 ? ~0ull : ((1ull << len) - 1)) << t;
            const bool match = len >= MATCH_MIN && (falls & block) == 0;
            if ((gheads >> t) & 1ull) {
                if (t >= singles_until) {
                    if (wide_mode) {
                        wide_flush(wide, nw, out, base, grp, cap);
                        wide_mode = false;
                        nw = 0;
                    } else if (lane < n_open && base + o.cid < cap) {
                        lane_nam_store(out, base + o.cid, grp, o);
                    }
                    base += gcnt;
                    gcnt = 0;
                    n_open = 0;
                }
                grp = readlane_u32(c_rsd, t);
            }
            if (!wide_mode) {
                if (len > 1 && t >= singles_until) {
                    uint32_t n_new = 0;
                    int my_hit = -1;  // the block hit (chunk lane) this lane takes or opens with
                    bool fits = true;
                    if (n_open == 0) {
                        n_new = len;  // a group's first block opens a NAM a hit
                        my_hit = lane < len ? (int)(t + lane) : -1;
                    } else if (match) {
                        uint64_t took;
                        my_hit = match_block(B, t, len, block, lane < n_open && o.qp < qs && qs <= o.qe, o.qe, o.rp,
                                             o.re, took);
                        const uint64_t opens = block & ~took;
                        n_new = (uint32_t)__popcll(opens);
                        fits = n_open + n_new <= 64;
                        // the k-th hit that opens a NAM goes to lane n_open + k
                        if (fits && n_new) {
                            if (lane_bit(opens)) B.hold[n_open + mbcnt(opens)] = lane;
                            wave_sync();
                            if (lane >= n_open && lane < n_open + n_new) my_hit = (int)B.hold[lane];
                            wave_sync();
                        }
                    } else {
                        uint64_t taken = 0;
                        for (uint32_t i = t; i < t + len; i++) {
                            const int hrs = (int)readlane_u32(c_rs, i);
                            const int hre = (int)readlane_u32(c_re, i);
                            const int hqe = (int)(readlane_u32(c_q, i) >> 16);
                            bool hext = false;
                            const bool hacc =
                                lane < n_open && nam_accepts(o.qp, o.qe, o.rp, o.re, qs, hqe, hrs, hre, hext);
                            const uint64_t avail = ballot(hacc) & ~taken;
                            if (!avail && n_open + n_new == 64) {
                                fits = false;
                                break;
                            }
                            const uint32_t win = avail ? (uint32_t)__builtin_ctzll(avail) : n_open + n_new;
                            taken |= avail ? (1ull << win) : 0ull;
                            n_new += avail ? 0u : 1u;
                            my_hit = lane == win ? (int)i : my_hit;
                        }
                    }
                    if (fits) {
                        const int src = my_hit < 0 ? 0 : my_hit;
                        const int4 hh = B.h[src];
                        const int hrs = hh.x, hre = hh.y, hqe = hh.z;
                        const bool take = my_hit >= 0 && lane < n_open;
                        const bool mk = my_hit >= 0 && lane >= n_open;
                        const bool grow = mk || (take && hqe > o.qe && hre > o.re);
                        o.qs = mk ? qs : o.qs;
                        o.rs = mk ? hrs : o.rs;
                        o.qe = grow ? hqe : o.qe;
                        o.re = grow ? hre : o.re;
                        o.qp = take || mk ? qs : o.qp;
                        o.rp = take || mk ? hrs : o.rp;
                        o.n = mk ? 1 : o.n + (take ? 1 : 0);
                        o.cid = mk ? gcnt + (lane - n_open) : o.cid;
                        n_open += n_new;
                        gcnt += n_new;
                        t += len;
                        continue;
                    }
                    singles_until = t + len;
                }
                // one hit
                const int rs = (int)readlane_u32(c_rs, t), re = (int)readlane_u32(c_re, t), qe = (int)(q >> 16);
                const uint64_t xq = ballot(qe > o.qe), xr = ballot(re > o.re);
                uint64_t free = n_open < 64 ? 1ull << n_open : 0ull, mk;
                const uint64_t acc = (free - 1) & ballot(o.qp < qs) & ballot(qs <= o.qe) & ballot(o.rp < rs) &
                                     ballot(rs <= o.re) & ~(xq ^ xr);
                if (acc == 0 && n_open == 64) {
                    n_open = retire_lanes(o, qs, out, base, grp, cap);
                    free = n_open < 64 ? 1ull << n_open : 0ull;
                }
                if (acc || n_open < 64) {
                    o.n = lane < n_open ? o.n : 0;
                    lanes_take(o, acc, xq & xr, free, mk, gcnt, qs, qe, rs, re);
                    n_open += mk ? 1u : 0u;
                    gcnt += mk ? 1u : 0u;
                    t++;
                    continue;
                }
                if (!wide.near && !wide.far) return MERGE_OVERFLOW;
                // the group continues on the wide list, in creation order, with
                // this hit and the rest of its block
                wput(wide, lane, WideNam{o.qs, o.qe, o.qp, o.rs, o.re, o.rp, (uint32_t)o.n, o.cid});
                nw = 64;
                wide_mark = 64;
                wide_mode = true;
                n_open = 0;
                singles_until = 0;
                if (box && box_cap) {
                    const int lo = wave_imin(o.rp), hi = wave_imax(o.re);
                    if (lane == 0) box[0] = ChunkBox{lo, hi};
                }
                wave_sync_mem();
            }
            // Wide form: going through the list's chunks in order and, inside a
            // chunk, through the block's pending hits in order gives each hit
            // the entry it would take hit by hit (the hits a chunk leaves
            // pending find no acceptor in it, by induction over the chunks),
            // and a chunk is read once per block instead of once per hit.
            uint64_t pend = block;
            const uint32_t nch = (nw + 63) >> 6;
            const bool boxed = box && nch <= box_cap;
            const int my_rs = (int)c_rs;
            for (uint32_t c = 0; c < nch && pend; c++) {
                // the pending hits the chunk's bounds admit (all of them
                // without bounds); the bounds of the chunk's start hold
                // for every entry that has not taken a hit of the block
                uint64_t cm = pend;
                if (boxed) {
                    const ChunkBox bx = box[c];
                    cm = ballot(bx.lo < my_rs && my_rs <= bx.hi) & pend;
                }
                if (!cm) continue;
                const uint32_t e = c * 64 + lane;
                const bool valid = e < nw;
                WideNam w{};
                if (valid) w = wget(wide, e);
                uint64_t taken = 0;
                int my_hit = -1;  // the hit (chunk lane) this entry takes
                if (match) {
                    my_hit = match_block(B, t, len, cm, valid && w.qp < qs && qs <= w.qe, w.qe, w.rp, w.re, taken);
                    pend &= ~taken;
                    cm = 0;
                }
                while (cm) {
                    const uint32_t i = (uint32_t)__builtin_ctzll(cm);
                    cm &= cm - 1;
                    const int hrs = (int)readlane_u32(c_rs, i);
                    const int hre = (int)readlane_u32(c_re, i);
                    const int hqe = (int)(readlane_u32(c_q, i) >> 16);
                    bool ext = false;
                    const bool acc = valid && nam_accepts(w.qp, w.qe, w.rp, w.re, qs, hqe, hrs, hre, ext);
                    const uint64_t bal = ballot(acc) & ~taken;
                    if (bal) {
                        const uint64_t win = bal & (0 - bal);
                        taken |= win;
                        my_hit = lane_bit(win) ? (int)i : my_hit;
                        pend &= ~(1ull << i);
                    }
                }
                if (taken) {
                    const int src = my_hit < 0 ? 0 : my_hit;
                    const int4 hh = B.h[src];
                    const int hrs = hh.x, hre = hh.y, hqe = hh.z;
                    const bool tk = my_hit >= 0;
                    const bool ext = tk && hqe > w.qe && hre > w.re;
                    if (ext) {
                        w.qe = hqe;
                        w.re = hre;
                    }
                    if (tk) {
                        w.qp = qs;
                        w.rp = hrs;
                        w.n++;
                    }
                    if (boxed) {
                        const int hi = wave_imax(ext ? hre : (int)0x80000000);
                        if (lane == 0 && box[c].hi < hi) box[c].hi = hi;
                    }
                    if (tk) wput(wide, e, w);
                    wave_sync_mem();
                }
            }
            // the hits no entry took open entries, in hit order, all at once
            if (pend) {
                if (nw >= 2 * wide_mark) {
                    // retire the dead entries (query_end before this block), keeping the order
                    uint32_t kept = 0;
                    for (uint32_t c0 = 0; c0 < nw; c0 += 64) {
                        const uint32_t e = c0 + lane;
                        WideNam w{};
                        bool keep = false;
                        if (e < nw) {
                            w = wget(wide, e);
                            keep = w.qe >= qs;
                            if (!keep && base + w.cid < cap) lane_nam_store(out, base + w.cid, grp, from_wide(w));
                        }
                        const uint64_t kb = ballot(keep);
                        wave_sync_mem();
                        if (keep) wput(wide, kept + mbcnt(kb), w);
                        kept += (uint32_t)__popcll(kb);
                        wave_sync_mem();
                    }
                    nw = kept;
                    wide_mark = kept > 64 ? kept : 64;
                    if (box && ((nw + 63) >> 6) <= box_cap) boxes_rebuild(wide, nw, box);
                    wave_sync_mem();
                }
                const uint32_t k = (uint32_t)__popcll(pend), at = nw + mbcnt(pend);
                const bool mine = lane_bit(pend);
                if (mine)
                    wput(wide, at, WideNam{qs, (int)(c_q >> 16), qs, (int)c_rs, (int)c_re, (int)c_rs, 1u,
                                           gcnt + mbcnt(pend)});
                // bounds of the one or two chunks the new entries lie in (only
                // while every chunk has them)
                const uint32_t c_last = (nw + k - 1) >> 6;
                if (box && c_last < box_cap) {
                    for (uint32_t c = nw >> 6; c <= c_last; c++) {
                        const bool in = mine && (at >> 6) == c;
                        const int lo = wave_imin(in ? (int)c_rs : 0x7fffffff);
                        const int hi = wave_imax(in ? (int)c_re : (int)0x80000000);
                        if (lane == 0) {
                            const bool begun = c == nw >> 6 && (nw & 63) != 0;
                            const ChunkBox bx = box[c];
                            box[c] = ChunkBox{begun ? min(bx.lo, lo) : lo, begun ? max(bx.hi, hi) : hi};
                        }
                    }
                }
                nw += k;
                gcnt += k;
                wave_sync_mem();
            }
            t += len;
        }
    }
    if (wide_mode) wide_flush(wide, nw, out, base, grp, cap);
    else if (lane < n_open && base + o.cid < cap) lane_nam_store(out, base + o.cid, grp, o);
    return base + gcnt;
}

struct MergeLds {
    DevHit hits[MERGE_LDS];
};

// reads whose (strand, ref) groups merge on waves of their own (k_merge_groups,
// then k_merge_split_finish): those that do not merge in arrival order. k_merge
// only groups them, so that its few long merges and those of k_merge_groups run
// side by side (100 003 reads of a repeat-rich genome: k_merge 185 us with the
// merges of up to 512 hits, now 76; k_merge_groups, as long as its largest group
// of 1590 hits, 219 us before and after, with long items first)
constexpr uint32_t MERGE_SPLIT = 0xfffffffdu;
// hits of one k_merge_groups work item: consecutive small groups of a split
// read merge on one wave
constexpr uint32_t ITEM_HITS = 384;
// reads of up to this many hits are tried in arrival order first
constexpr uint32_t ARRIVAL_MAX = 512;
// entries of a wide list that lie in LDS: per wave of k_merge, and per group of
// k_merge_groups (one wave per block)
constexpr int MERGE_WIDE_LDS = 128;
constexpr int GROUP_WIDE_LDS = 512;
// chunk bounds of a k_merge_groups wide list (lists up to 8,192 entries)
constexpr uint32_t GROUP_BOXES = 128;

// the reads that k_merge4 handed on, one per wave, and one wave per block: waves
// take very different times, and a block holds its LDS (for groups and wide lists)
// until its slowest is done
__global__ __launch_bounds__(64) void k_merge(DevBatch b) {
    __shared__ uint64_t lkeys[MERGE_LDS];
    __shared__ WideNam lwide[MERGE_WIDE_LDS];  // the wide list of reads with few enough hits
    __shared__ BlockLds lblock;
    const uint32_t lane = lane_id();
    if (hits_missing(b)) return;
    const uint32_t cnt = sload(&b.ctl->n_sel[SEL_DEFERRED]);
    for (uint32_t w = blockIdx.x; w < cnt; w += gridDim.x) {
        const uint32_t r = uni32(b.sel_ids[(uint64_t)b.n_reads + w]);
        const bool rescue = (uni32(b.flags[r]) & GIS_FLAG_RESCUED) != 0;
        const uint64_t hb = uni64(rescue ? b.rhit_off[r] : b.hit_off[r]);
        const uint32_t nh = uni32(rescue ? b.rhit_total[r] : b.hit_total[r]);
        const DevHit *ghits = (rescue ? b.rhits : b.hits) + hb;
        gis_nam *fin = (rescue ? b.rnam_fin : b.nam_fin) + hb;
        uint64_t *gkeys = b.merge_scratch ? (rescue ? b.rkeys : b.keys) + 2 * hb : nullptr;
        uint32_t total = nh <= ARRIVAL_MAX ? merge_arrival<true>(ghits, nh, fin, nh) : MERGE_OVERFLOW;
        if (total == MERGE_OVERFLOW && b.merge_scratch) {
            // group the hits; k_merge_groups merges them, a large group a wave
            uint32_t *bins = reinterpret_cast<uint32_t *>(lkeys);
            bool binned;
            const uint64_t *ord = group_order(nh, ghits, gkeys, gkeys + nh, bins, binned);
            const uint32_t code = ord == nullptr ? 0u : (ord == gkeys ? 1u : 2u);
            uint64_t *slots = code == 1u ? gkeys + nh : gkeys;
            // work items: runs of consecutive groups of at least ITEM_HITS hits (a
            // larger group is an item of its own); each item's start goes to
            // slots[item], which later holds its NAM count
            uint32_t K = 0, cur = 0;
            // start: of a lane's group where head, growing with the lane
            auto cut = [&](uint64_t heads, uint32_t start) {
                for (;;) {
                    heads &= ballot(start >= cur + ITEM_HITS);
                    if (!heads) break;
                    if (lane == 0) slots[K] = (uint64_t)cur << 32;
                    K++;
                    cur = readlane_u32(start, (uint32_t)__builtin_ctzll(heads));
                }
            };
            if (binned) {
                uint32_t done = 0;
                for (uint32_t d0 = 0; d0 < 256; d0 += 64) {
                    const uint32_t end = bins[d0 + lane];
                    const uint32_t start = (uint32_t)__builtin_amdgcn_update_dpp((int)done, (int)end, 0x138, 0xf, 0xf, false);
                    done = readlane_u32(end, 63);
                    cut(ballot(end > start), start);
                }
            } else {
                uint32_t before = 0;
                each_ahead<uint32_t>(nh, [&](uint32_t i) {
                    return ord ? (uint32_t)(ord[i] >> 32) : ghits[i].ref_strand;  // (the group above the index)
                }, [&](uint32_t i, uint32_t grp) {
                    const uint32_t prev =
                        (uint32_t)__builtin_amdgcn_update_dpp((int)before, (int)grp, 0x138, 0xf, 0xf, false);
                    before = readlane_u32(grp, 63);
                    cut(ballot(i > 0 && i < nh && prev != grp), i);
                });
            }
            if (lane == 0) slots[K] = (uint64_t)cur << 32;
            K++;
            wave_sync_mem();
            {
                // long items from the list's front, the others from its back
                for (uint32_t g0 = 0; g0 < K; g0 += 64) {
                    const uint32_t g = g0 + lane;
                    uint32_t gs = 0, ge = 0;
                    if (g < K) {
                        gs = (uint32_t)(slots[g] >> 32);
                        ge = g + 1 < K ? (uint32_t)(slots[g + 1] >> 32) : nh;
                    }
                    const uint64_t lm = ballot(ge - gs >= 2 * ITEM_HITS), sm = ballot(g < K) & ~lm;
                    uint32_t at_l = 0, at_s = 0;
                    if (lane == 0) {
                        if (lm) at_l = atomicAdd(&b.ctl->n_gwork[0], (uint32_t)__popcll(lm));
                        if (sm) at_s = atomicAdd(&b.ctl->n_gwork[1], (uint32_t)__popcll(sm));
                    }
                    at_l = uni32(at_l) + mbcnt(lm);
                    at_s = uni32(at_s) + mbcnt(sm);
                    if (g < K)
                        b.gwork[lane_bit(lm) ? at_l : b.gwork_cap - 1 - at_s] = make_uint4(r, gs, ge, g | (code << 30));
                }
                if (lane == 0) {
                    const uint32_t si = atomicAdd(&b.ctl->n_split, 1u);
                    b.split_list[si] = make_uint4(r, K, code, 0u);
                    b.nam_cnt[r] = MERGE_SPLIT;
                }
                wave_sync_mem();
                continue;
            }
        }
        if (total == MERGE_OVERFLOW && nh <= (uint32_t)MERGE_LDS) {
            // no scratch (yet): here, group by group, with a wide list (NAMs <= hits)
            bool binned;
            const uint64_t *ord = group_order(nh, ghits, lkeys, nullptr, reinterpret_cast<uint32_t *>(lkeys), binned);
            const WideList wl{(LdsWideNam *)lwide, nullptr, (uint32_t)MERGE_WIDE_LDS};
            total = merge_range(ghits, ord, 0, nh, wl, fin, nh, lblock);
        }
        if (total == MERGE_OVERFLOW) {
            // needs the global scratch, which this run does not have yet
            if (lane == 0) {
                atomicOr(&b.ctl->overflow, OVF_MERGE);
                b.nam_cnt[r] = 0;
            }
            continue;
        }
        if (lane == 0) b.nam_cnt[r] = total;
        wave_sync_mem();
    }
}

// one wave per work item (a run of consecutive groups of a split read): its
// hits (in grouped order) merge into NAMs at the item's own hit-indexed region
// of the read's output; the NAM count goes to the read's item slot
__global__ __launch_bounds__(64) void k_merge_groups(DevBatch b) {
    __shared__ WideNam lwide[GROUP_WIDE_LDS];
    __shared__ ChunkBox lbox[GROUP_BOXES];
    __shared__ BlockLds lblock;
    const uint32_t lane = lane_id();
    // (long items first: the kernel is as long as the last of them)
    const uint32_t n_long = sload(&b.ctl->n_gwork[0]), cnt = n_long + sload(&b.ctl->n_gwork[1]);
    for (uint32_t w = blockIdx.x; w < cnt; w += gridDim.x) {
        const uint4 it = b.gwork[w < n_long ? w : b.gwork_cap - 1 - (w - n_long)];
        const uint32_t r = it.x, gs = it.y, ge = it.z, g = it.w & 0x3fffffffu, code = it.w >> 30;
        const bool rescue = (b.flags[r] & GIS_FLAG_RESCUED) != 0;
        const uint64_t hb = rescue ? b.rhit_off[r] : b.hit_off[r];
        const uint32_t nh = rescue ? b.rhit_total[r] : b.hit_total[r];
        uint64_t *gkeys = (rescue ? b.rkeys : b.keys) + 2 * hb;
        const uint64_t *ord = code == 0u ? nullptr : (code == 1u ? gkeys : gkeys + nh);
        uint64_t *slots = code == 1u ? gkeys + nh : gkeys;
        const DevHit *ghits = (rescue ? b.rhits : b.hits) + hb;
        // the first GROUP_WIDE_LDS wide entries in LDS, the rest in the
        // group's global region (as many entries as hits)
        WideNam *far = (rescue ? b.rnam_ws : b.nam_ws) + hb + gs;
        gis_nam *out = (rescue ? b.rnam_fin : b.nam_fin) + hb + gs;
        const WideList wl{(LdsWideNam *)lwide, far, (uint32_t)GROUP_WIDE_LDS};
        const uint32_t c = merge_range(ghits, ord, gs, ge, wl, out, ge - gs, lblock, lbox, GROUP_BOXES);
        if (lane == 0) slots[g] = ((uint64_t)gs << 32) | c;
        wave_sync_mem();
    }
}

// one wave per split read: the groups' NAMs move to consecutive places in
// group order (canonical order) with nam_id = rank
__global__ __launch_bounds__(64 * WPB) void k_merge_split_finish(DevBatch b) {
    const uint32_t lane = lane_id();
    const unsigned int cnt = sload(&b.ctl->n_split);
    for (uint32_t w = blockIdx.x * WPB + (threadIdx.x >> 6); w < cnt; w += gridDim.x * WPB) {
        const uint4 e = b.split_list[w];
        const uint32_t r = e.x, G = e.y, code = e.z;
        const bool rescue = (b.flags[r] & GIS_FLAG_RESCUED) != 0;
        const uint64_t hb = rescue ? b.rhit_off[r] : b.hit_off[r];
        const uint32_t nh = rescue ? b.rhit_total[r] : b.hit_total[r];
        uint64_t *gkeys = (rescue ? b.rkeys : b.keys) + 2 * hb;
        const uint64_t *slots = code == 1u ? gkeys + nh : gkeys;
        gis_nam *fin = (rescue ? b.rnam_fin : b.nam_fin) + hb;
        // base <= gs: every NAM moves towards the front, and nothing is moved onto
        // what a later step reads, so each step's 128 NAMs are loaded before the
        // one before it stores (a lone wave waits for its loads); the first item's
        // are in place
        const uint64_t some = lane < G ? slots[lane] : 0;
        auto slot = [&](uint32_t g) { return g < 64 ? readlane_u64(some, g) : uni64(slots[g]); };
        uint32_t g = 0, c0 = 0, base = (uint32_t)slot(0);
        uint32_t gs = 0, c = 0;
        auto step = [&](gis_nam (&x)[2]) {  // loads the next step's; false at the end
            c0 += 128;
            while (c0 >= c) {
                base += g > 0 ? c : 0;
                if (++g >= G) return false;
                const uint64_t sg = slot(g);
                gs = (uint32_t)(sg >> 32);
                c = (uint32_t)sg;
                c0 = 0;
                if (c) break;
            }
#pragma unroll
            for (uint32_t u = 0; u < 2; u++)
                if (c0 + 64 * u + lane < c) x[u] = fin[gs + c0 + 64 * u + lane];
            return true;
        };
        auto store = [&](gis_nam (&x)[2], uint32_t at, uint32_t n) {
            wave_sync_mem();
#pragma unroll
            for (uint32_t u = 0; u < 2; u++) {
                const uint32_t k = 64 * u + lane;
                if (k < n) {
                    x[u].nam_id = (int32_t)(at + k);
                    fin[at + k] = x[u];
                }
            }
        };
        gis_nam x[2], y[2];
        bool more = step(x);
        while (more) {
            const uint32_t at = base + c0, n = min(128u, c - c0);
            more = step(y);
            store(x, at, n);
            if (!more) break;
            const uint32_t at2 = base + c0, n2 = min(128u, c - c0);
            more = step(x);
            store(y, at2, n2);
        }
        if (lane == 0) b.nam_cnt[r] = base;
        wave_sync_mem();
    }
}

// ---------------------------------------------------------------------------
// Merge of four reads per wave (16 lanes each) for reads with at most 64
// hits. Each lane holds one NAM of its read; NAMs of every (strand, ref)
// group of the current strand share the segment, so the hits are taken in
// arrival order without grouping them: within one group that is
// (query_start, ref_start) order, and a NAM only accepts hits of its own
// group. Each segment broadcasts its read's next hit from LDS, a ballot
// restricted to the segment picks the first accepting NAM (creation order),
// and a hit nobody accepts opens a NAM in the segment's next lane. When a
// strand's hits end, its NAMs are final: each lane ranks its NAM among the
// segment's by (ref_id, creation index), which is canonical order within the
// strand, and writes it. A read with more than 16 NAMs on one strand is merged
// again by the whole wave (merge_arrival; 64 hits make at most 64 NAMs), and a
// read of more than 64 hits is listed for k_merge.

constexpr uint32_t SEG = 16;
constexpr uint32_t RPW = 64 / SEG;

// The NAMs of the segments for which `on` holds (those of their lanes that took
// hits) at out + base, ranked by (ref_id, creation index = lane). A segment is
// one DPP row of 16 lanes: rotating the row by 1..15 shows each lane every
// other lane's key. Lanes are below 16, so no key is all ones, which marks the
// free lanes.
__device__ __forceinline__ void seg_finalize(gis_nam *out, uint32_t base, uint32_t j, uint32_t rsd, const LaneNam &o,
                                             bool on) {
    const uint32_t key = ((rsd & 0x7fffffffu) << 8) | j;
    const int kv = (int)(o.n > 0 ? key : 0xffffffffu);
    uint32_t rank = 0;
#define GIS_ROW_ROR(r) rank += (uint32_t)__builtin_amdgcn_mov_dpp(kv, 0x120 + (r), 0xf, 0xf, true) < key ? 1u : 0u
    GIS_ROW_ROR(1); GIS_ROW_ROR(2); GIS_ROW_ROR(3); GIS_ROW_ROR(4); GIS_ROW_ROR(5);
    GIS_ROW_ROR(6); GIS_ROW_ROR(7); GIS_ROW_ROR(8); GIS_ROW_ROR(9); GIS_ROW_ROR(10);
    GIS_ROW_ROR(11); GIS_ROW_ROR(12); GIS_ROW_ROR(13); GIS_ROW_ROR(14); GIS_ROW_ROR(15);
#undef GIS_ROW_ROR
    if (on && o.n > 0) lane_nam_store(out, base + rank, rsd, o);
}

// The hits of one strand of each segment's read (cnt of them from hits on, in
// LDS) merged into the segment's lanes. Returns the read's hits that found a
// lane (fewer than cnt: the strand needs more than 16 NAMs).
__device__ __forceinline__ uint32_t seg_merge(const DevHit *hits, uint32_t cnt, LaneNam &o, uint32_t &rsd_o) {
    constexpr uint64_t FIRST = 0x0001000100010001ull;  // lane 0 of each row
    uint64_t free = FIRST;  // the lane of each row that opens the next NAM (none when the row is full)
    const uint32_t most = wave_max_dpp(cnt), last = cnt ? cnt - 1 : 0;
    for (uint32_t t = 0; t < most; t++) {
        const uint4 h = reinterpret_cast<const uint4 *>(hits)[min(t, last)];
        const int rs = (int)h.y, re = (int)h.z, qs = (int)(h.w & 0xffffu), qe = (int)(h.w >> 16);
        const uint64_t xq = ballot(qe > o.qe), xr = ballot(re > o.re);
        const uint64_t acc = ballot(rsd_o == h.x) & ballot(o.qp < qs) & ballot(qs <= o.qe) & ballot(o.rp < rs) &
                             ballot(rs <= o.re) & ~(xq ^ xr);
        // the first accepting lane of the segment takes the hit; else the
        // segment's free lane opens a NAM with it
        const uint64_t me = first_of_rows((acc | free) & ballot(t < cnt)), mk = me & free;
        const bool b_mk = lane_bit(mk), b_end = lane_bit(mk | (me & xq & xr)), b_me = lane_bit(me);
        free = (free ^ mk) | ((mk << 1) & ~FIRST);
        o.qs = b_mk ? qs : o.qs;
        o.rs = b_mk ? rs : o.rs;
        rsd_o = b_mk ? h.x : rsd_o;
        o.qe = b_end ? qe : o.qe;
        o.re = b_end ? re : o.re;
        o.qp = b_me ? qs : o.qp;
        o.rp = b_me ? rs : o.rp;
        o.n += b_me ? 1 : 0;
    }
    return row_sum((uint32_t)o.n);
}

// The four reads of a wave: hits points at this lane's read's hits in LDS (at
// least one may be read), nh and nf at their count and the count of forward
// ones, out at its NAMs. Returns the read's NAM count, or MERGE_OVERFLOW when a
// strand needs more than 16.
//
// Bound by VALU issue, so what can be a mask is one, on the scalar unit: the
// acceptance tests, the first accepting or else the free lane of each row, the
// free lanes. A lane's creation index is its place in the row. The two strands
// are independent: each read's longer one goes first, so that the wave's steps
// are the longest of four long strands plus the longest of four short ones,
// without a strand switch inside, and the NAMs are ranked and written twice a
// wave and not at every read's own switch. 65,536 reads of 23 hits: 51 -> 38 us.
__device__ __forceinline__ uint32_t merge_segments(const DevHit *hits, uint32_t nh, uint32_t nf, gis_nam *out) {
    const uint32_t j = lane_id() % SEG, nr = nh - nf;
    const bool rev = nr > nf;  // the reverse strand first
    LaneNam oa{0, 0, 0, 0, 0, 0, 0, 0}, ob{0, 0, 0, 0, 0, 0, 0, 0};
    uint32_t ra = 0xffffffffu, rb = 0xffffffffu;  // the lanes' groups
    uint32_t took = seg_merge(hits + (rev ? nf : 0u), rev ? nr : nf, oa, ra);
    took += seg_merge(hits + (rev || nr == 0 ? 0u : nf), rev ? nf : nr, ob, rb);
    const uint32_t ma = row_sum(oa.n > 0 ? 1u : 0u), mb = row_sum(ob.n > 0 ? 1u : 0u);
    const bool ok = took == nh;
    seg_finalize(out, rev ? mb : 0u, j, ra, oa, ok);
    seg_finalize(out, rev ? 0u : ma, j, rb, ob, ok);
    return ok ? ma + mb : MERGE_OVERFLOW;
}

__global__ __launch_bounds__(64 * WPB) void k_merge4(DevBatch b, ReadSet set) {
    __shared__ DevHit lh[WPB][RPW][64];
    const uint32_t lane = lane_id(), seg = lane / SEG, j = lane % SEG;
    const int wid = (int)uni32(threadIdx.x >> 6);
    if (hits_missing(b)) return;
    const uint32_t cnt = set_count(set);
    const uint32_t stride = gridDim.x * WPB * RPW;
    for (uint32_t w0 = wave_index(WPB) * RPW; w0 < cnt; w0 += stride) {
        const uint32_t widx = w0 + seg;
        const bool act = widx < cnt;
        uint32_t r = 0, nh = 0;
        uint64_t hb = 0;
        bool rescue = false;
        if (act) {
            r = set_at(set, widx);
            rescue = (b.flags[r] & GIS_FLAG_RESCUED) != 0;
            hb = rescue ? b.rhit_off[r] : b.hit_off[r];
            nh = rescue ? b.rhit_total[r] : b.hit_total[r];
        }
        const bool many = nh > 64;
        if (many) nh = 0;
        const DevHit *gh = (rescue ? b.rhits : b.hits) + hb;
        uint32_t fwd = 0;
        for (uint32_t k = j; k < nh; k += SEG) {
            const uint4 h = reinterpret_cast<const uint4 *>(gh)[k];
            reinterpret_cast<uint4 *>(lh[wid][seg])[k] = h;
            fwd += (h.x >> 31) ^ 1u;
        }
        const uint32_t nf = row_sum(fwd);
        wave_sync_mem();
        gis_nam *out = (rescue ? b.rnam_fin : b.nam_fin) + hb;
        const uint32_t total = merge_segments(lh[wid][seg], nh, nf, out);
        const bool ovf = total == MERGE_OVERFLOW;
        if (act && j == 0 && !many && !ovf) b.nam_cnt[r] = total;
        // a read with more than 16 NAMs on a strand has the whole wave
        uint64_t redo = ballot(ovf && j == 0);
        while (redo) {
            const uint32_t l = (uint32_t)__builtin_ctzll(redo);
            redo &= redo - 1;
            const uint32_t nl = readlane_u32(nh, l);
            gis_nam *ol = reinterpret_cast<gis_nam *>(
                (uint64_t)readlane_u32((uint32_t)(uintptr_t)out, l) |
                ((uint64_t)readlane_u32((uint32_t)((uintptr_t)out >> 32), l) << 32));
            const uint32_t all = merge_arrival(lh[wid][l / SEG], nl, ol, nl);
            if (lane == l) b.nam_cnt[r] = all;
        }
        // the reads handed on to k_merge
        const bool defer = many && j == 0;
        const uint64_t dm = ballot(defer);
        if (dm) {
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&b.ctl->n_sel[SEL_DEFERRED], (uint32_t)__popcll(dm));
            at = uni32(at);
            if (defer) b.sel_ids[(uint64_t)b.n_reads + at + mbcnt(dm)] = r;
        }
        wave_sync_mem();
    }
}

// ---------------------------------------------------------------------------
// fused: the whole path of one read in one wave. Each lane holds randstrobe
// pair i (forward i, reverse complement i) in registers, so a read fits when
// it has at most 64 + w_min syncmers; hits and the merge live in LDS. Reads
// beyond these limits are appended to the spill list for the per-stage
// kernels.
//
// The kernel is persistent over a device work queue: a list of read ids
// ordered by length (longest first), cut by the host into a long and a short
// bin that run as separate launches with their own LDS tiling (LMAX). Waves
// take reads either statically (wave w takes queue entries w, w + W, ...,
// which deals the length-sorted queue round robin) or dynamically (a wave
// grabs `chunk` entries at a time from a counter in the control block).

constexpr int F_SYCAP = 96;
static_assert(F_SYCAP <= 160, "the syncmer hashes take the s-mer hashes' place");

template <int LMAX>
struct alignas(8) FusedSeedLds {
    uint64_t sh[LMAX];  // then the syncmers' hashes
    uint64_t nmask[LMAX / 64 + 2];
    uint64_t pk[2 * ((LMAX + 63) / 64) + 1];
    uint16_t sy_pos[F_SYCAP];
    uint8_t st[LMAX];
};

template <int LMAX>
union alignas(16) FusedLds {
    FusedSeedLds<LMAX> seed;
    MergeLds merge;
};

// hand read r to the per-stage kernels (reads spill rarely, so one atomic
// per spilled read does not contend)
__device__ __forceinline__ void spill_read(const DevBatch &b, uint32_t r) {
    if (lane_id() == 0) {
        b.flags[r] = FLAG_SPILL;
        b.nam_cnt[r] = 0;
        b.hit_total[r] = 0;
        b.rhit_total[r] = 0;
        const unsigned int at = atomicAdd(&b.ctl->n_spill, 1u);
        b.spill_ids[at] = r;
    }
    wave_sync_mem();
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The bucket line of one query randstrobe, fetched in one round trip. The
// empty asm takes every loaded word, so all eight loads issue before the
// first wait: otherwise the compiler sinks the record loads into the
// small-bucket branch, behind the wait for the bucket's bounds, and each
// probe pays two dependent fetches. Each lane holds one query randstrobe,
// so a read's forward and reverse-complement lines arrive together.
__device__ __forceinline__ void probe_line_now(const DevIndex &ix, Probe &P) {
    const u32x4 *l = reinterpret_cast<const u32x4 *>(ix.lines) +
                     (uint64_t)(uint32_t)(P.key >> (64 - ix.bits)) * BUCKET_LINE;
    u32x4 a[BUCKET_LINE];
#pragma unroll
    for (uint32_t j = 0; j < BUCKET_LINE; j++) a[j] = l[j];
    asm volatile("" ::"v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]));
    P.s = (uint64_t)a[0].x | ((uint64_t)a[0].y << 32);
    P.e = P.s + a[0].z;
#pragma unroll
    for (uint32_t j = 0; j < PROBE_SMALL; j++)
        P.r[j] = IdxRec{(uint64_t)a[j + 1].x | ((uint64_t)a[j + 1].y << 32), a[j + 1].z, a[j + 1].w};
}

// find + is_filtered + the counting run walk of one query randstrobe through
// its fetched bucket line (the per-stage lookup's probe): position, found
// and not filtered, kept hits, and for a small bucket the kept records' mask
__device__ __forceinline__ void fused_probe(const DevIndex &ix, Probe &P, int qs, int qe, uint64_t &pos,
                                            bool &good, uint32_t &kept, uint32_t &mask, bool &small) {
    probe_finish(ix, P, qs, qe);
    pos = P.pos;
    good = P.found && !P.filtered;
    kept = P.hc;
    mask = P.keep;
    small = probe_small(P);
}

// the records of a small bucket's line that `mask` selects, written as hits
// in run order (the line is read again; it was fetched by the probe)
__device__ __forceinline__ void fused_emit_line(const DevIndex &ix, uint64_t key, uint32_t mask, int qs, int qe,
                                                uint32_t strand_bit, DevHit *out) {
    Probe P;
    P.key = key;
    probe_line(ix, P);
    P.keep = mask;
    probe_emit(ix, P, qs, qe, strand_bit, out);
}

// The lanes' runs flagged in `mine` walked by the whole wave, one after the
// other: the kept count goes to the owning lane's `kept`, and with out the
// hits go to out + (the owning lane's at), with the owning lane's strand bit.
__device__ __forceinline__ void fused_wave_walks(const DevIndex &ix, bool mine, uint64_t pos, uint64_t key,
                                                 uint32_t qs, uint32_t qe, uint32_t strand_bit, uint32_t &kept,
                                                 DevHit *out, uint32_t at) {
    const uint32_t lane = lane_id();
    uint64_t m = ballot(mine);
    while (m) {
        const uint32_t l = (uint32_t)__builtin_ctzll(m);
        m &= m - 1;
        const uint64_t pl =
            (uint64_t)readlane_u32((uint32_t)pos, l) | ((uint64_t)readlane_u32((uint32_t)(pos >> 32), l) << 32);
        const uint64_t kl =
            (uint64_t)readlane_u32((uint32_t)key, l) | ((uint64_t)readlane_u32((uint32_t)(key >> 32), l) << 32);
        const uint32_t k = walk_run_wave(ix, pl, kl, (int)readlane_u32(qs, l), (int)readlane_u32(qe, l),
                                         readlane_u32(strand_bit, l), out ? out + readlane_u32(at, l) : nullptr);
        if (lane == l) kept = k;
    }
}

// One read through seeding, lookup and its hits. With `stash` (an LDS slot
// of 64 hits), a read with 1 to 64 hits leaves them there and reports their
// count in stashed for a merge with three other reads (fused_quad_merge);
// every other read is merged alone (or spilled) here.
template <int LMAX>
__device__ __forceinline__ void fused_read(const DevBatch &b, const DevIndex &ix, const SeedParams &P,
                                           FusedLds<LMAX> &S, uint32_t r, uint32_t rescue_cutoff,
                                           uint32_t hard_cutoff, DevHit *stash, uint32_t &stashed,
                                           uint32_t &stashed_fwd) {
    stashed = 0;
    const uint32_t lane = lane_id();
    const int L = (int)sload(b.read_len + r);
    bool spill = L > LMAX;
    uint32_t nh = 0, n_fwd = 0, nh_fwd = 0;
    bool rescue = false;
    float frac = 1.0f;
    if (!spill) {
        SeedBufs B{S.seed.pk, S.seed.st, S.seed.sh, S.seed.sh, S.seed.sy_pos, S.seed.nmask};
        const uint32_t n = seed_syncmers(b.seqs + sload(b.read_off + r), L, P, B, F_SYCAP, nullptr, nullptr);
        n_fwd = ((uint32_t)L >= P.w_max && n > P.w_min) ? n - P.w_min : 0;
        spill = n > (uint32_t)F_SYCAP || n_fwd > 64;
        // query randstrobe j (randstrobes_query order: the forward ones, then
        // the reverse-complement ones) on lane j, and randstrobe 64 + j, when
        // the read has more than 64, on lane j's second slot
        const uint32_t nq = 2 * n_fwd;
        const bool aa = !spill && lane < nq, ab = !spill && lane + 64 < nq;
        Rs1 qa{}, qb{};
        if (aa) qa = randstrobe_one(B, n, n_fwd, lane, L, P);
        if (ab) qb = randstrobe_one(B, n, n_fwd, lane + 64, L, P);
        wave_sync();  // the syncmer lists are dead from here; LDS becomes MergeLds
        if (!spill) {
            // each randstrobe through find / filter / run walk: the
            // bucket-line probe of the per-stage lookup; a small bucket's kept
            // records are remembered as a mask over its line. Second-slot
            // randstrobes (64 and up, n_fwd <= 64) are all reverse-complement.
            const uint32_t sba = lane < n_fwd ? 0u : 0x80000000u, sbb = 0x80000000u;
            uint64_t pa = GIS_NOT_FOUND, pb = GIS_NOT_FOUND;
            uint32_t ha = 0, hb = 0, ka = 0, kb = 0;
            bool ga = false, gb = false, sa = false, sb = false;
            // the second slot first: the first slot's probe then stays in
            // registers for the hits of a read that is not rescued
            if (ab) {
                Probe Q;
                Q.key = qb.h;
                probe_line_now(ix, Q);
                fused_probe(ix, Q, (int)qb.s, (int)qb.e, pb, gb, hb, kb, sb);
            }
            Probe QA;
            QA.key = qa.h;
            if (aa) {
                probe_line_now(ix, QA);
                fused_probe(ix, QA, (int)qa.s, (int)qa.e, pa, ga, ha, ka, sa);
            }
            // (the whole wave is active here: spill and rescue are wave-uniform)
            const uint32_t found = wave_count(pa != GIS_NOT_FOUND) + wave_count(pb != GIS_NOT_FOUND);
            const uint32_t good = wave_count(ga) + wave_count(gb);
            const uint32_t hits_norm = wave_sum_dpp(ha + hb);
            frac = found > 0 ? (float)good / (float)found : 1.0f;
            rescue = (double)frac < 0.7 || hits_norm == 0;
            if (!rescue) {
                // hits into LDS in query order (forward seeds, then reverse
                // ones): the first slot's straight from the lines its probes
                // fetched, a second slot's lines read again
                const uint32_t ia = wave_incl_scan_dpp(ha), ib = nq > 64 ? wave_incl_scan_dpp(hb) : 0u;
                const uint32_t tot_a = readlane_u32(ia, 63);
                nh_fwd = n_fwd ? readlane_u32(ia, n_fwd - 1) : 0u;
                nh = tot_a + readlane_u32(ib, 63);
                spill = nh > (uint32_t)MERGE_LDS;
                if (!spill) {
                    DevHit *dst = stash && nh <= 64 ? stash : S.merge.hits;
                    if (ha) probe_emit(ix, QA, (int)qa.s, (int)qa.e, sba, dst + (ia - ha));
                    if (hb) {
                        DevHit *ob = dst + tot_a + (ib - hb);
                        if (sb) fused_emit_line(ix, qb.h, kb, (int)qb.s, (int)qb.e, sbb, ob);
                        else walk_run(ix, pb, qb.h, (int)qb.s, (int)qb.e, sbb, ob);
                    }
                    wave_sync_mem();
                }
            } else {
                bool wa = false, wb = false;  // taken runs longer than WALK_WAVE_MIN: the wave walks them
                {
                    // run lengths, and the taken prefix of each strand: a seed's
                    // rank among its strand's seeds in (count, start, end) order
                    const uint32_t ca = aa && pa != GIS_NOT_FOUND ? dev_get_count(ix, pa) : 0u;
                    const uint32_t cb = ab && pb != GIS_NOT_FOUND ? dev_get_count(ix, pb) : 0u;
                    const bool fwd_a = lane < n_fwd;
                    uint32_t ranka = 0, rankb = 0;
                    for (uint32_t j = 0; j < n_fwd; j++) {
                        // forward randstrobe j (lane j) and reverse-complement
                        // randstrobe n_fwd + j (lane or second slot)
                        const uint32_t cf = readlane_u32(ca, j), sf = readlane_u32(qa.s, j), ef = readlane_u32(qa.e, j);
                        const uint32_t y = n_fwd + j;
                        const bool hi = y >= 64;
                        const uint32_t yl = hi ? y - 64 : y;
                        const uint32_t cr = hi ? readlane_u32(cb, yl) : readlane_u32(ca, yl);
                        const uint32_t sr = hi ? readlane_u32(qb.s, yl) : readlane_u32(qa.s, yl);
                        const uint32_t er = hi ? readlane_u32(qb.e, yl) : readlane_u32(qa.e, yl);
                        const uint32_t cj = fwd_a ? cf : cr, sj = fwd_a ? sf : sr, ej = fwd_a ? ef : er;
                        ranka += (cj > 0 && rh_less(cj, sj, ej, ca, qa.s, qa.e)) ? 1u : 0u;
                        rankb += (cr > 0 && rh_less(cr, sr, er, cb, qb.s, qb.e)) ? 1u : 0u;
                    }
                    const bool ta = ca > 0 && ca <= hard_cutoff && (ca <= rescue_cutoff || ranka < 5);
                    const bool tb = cb > 0 && cb <= hard_cutoff && (cb <= rescue_cutoff || rankb < 5);
                    wa = ta && ca > WALK_WAVE_MIN;
                    wb = tb && cb > WALK_WAVE_MIN;
                    ha = ta && !wa ? walk_run(ix, pa, qa.h, (int)qa.s, (int)qa.e, sba, nullptr) : 0u;
                    hb = tb && !wb ? walk_run(ix, pb, qb.h, (int)qb.s, (int)qb.e, sbb, nullptr) : 0u;
                    fused_wave_walks(ix, wa, pa, qa.h, qa.s, qa.e, sba, ha, nullptr, 0u);
                    fused_wave_walks(ix, wb, pb, qb.h, qb.s, qb.e, sbb, hb, nullptr, 0u);
                }
                // hits into LDS in query order: forward seeds, then reverse ones
                const uint32_t ia = wave_incl_scan_dpp(ha), ib = nq > 64 ? wave_incl_scan_dpp(hb) : 0u;
                const uint32_t tot_a = readlane_u32(ia, 63);
                nh_fwd = n_fwd ? readlane_u32(ia, n_fwd - 1) : 0u;
                nh = tot_a + readlane_u32(ib, 63);
                spill = nh > (uint32_t)MERGE_LDS;
                if (!spill) {
                    // a read that goes to the four-read merge writes its hits
                    // straight into its stash slot
                    DevHit *dst = stash && nh <= 64 ? stash : S.merge.hits;
                    const uint32_t oa = ia - ha, ob = tot_a + ib - hb;
                    // a taken seed of a small bucket keeps the records the probe
                    // kept (its run walk is the same in both modes)
                    if (ha && !wa) {
                        if (sa) fused_emit_line(ix, qa.h, ka, (int)qa.s, (int)qa.e, sba, dst + oa);
                        else walk_run(ix, pa, qa.h, (int)qa.s, (int)qa.e, sba, dst + oa);
                    }
                    if (hb && !wb) {
                        if (sb) fused_emit_line(ix, qb.h, kb, (int)qb.s, (int)qb.e, sbb, dst + ob);
                        else walk_run(ix, pb, qb.h, (int)qb.s, (int)qb.e, sbb, dst + ob);
                    }
                    uint32_t unused_a = 0, unused_b = 0;
                    fused_wave_walks(ix, wa, pa, qa.h, qa.s, qa.e, sba, unused_a, dst, oa);
                    fused_wave_walks(ix, wb, pb, qb.h, qb.s, qb.e, sbb, unused_b, dst, ob);
                    wave_sync_mem();
                }
            }
        }
    }
    if (spill) {
        spill_read(b, r);
        return;
    }
    if (stash && nh > 0 && nh <= 64) {
        // the hits are in the stash slot
        if (lane == 0) {
            b.frac[r] = frac;
            b.flags[r] = (uint8_t)((rescue ? GIS_FLAG_RESCUED : 0) | (n_fwd == 0 ? GIS_FLAG_NO_RANDSTROBES : 0));
            b.hit_total[r] = 0;
            b.rhit_total[r] = 0;
        }
        stashed = nh;
        stashed_fwd = nh_fwd;
        return;
    }
    uint32_t total = 0;
    if (nh > 0) total = merge_arrival(S.merge.hits, nh, b.nam_slots + (uint64_t)r * F_NAMCAP, (uint32_t)F_NAMCAP);
    if (total > (uint32_t)F_NAMCAP) {  // includes MERGE_OVERFLOW
        spill_read(b, r);
        return;
    }
    if (lane == 0) {
        b.frac[r] = frac;
        b.flags[r] = (uint8_t)((rescue ? GIS_FLAG_RESCUED : 0) | (n_fwd == 0 ? GIS_FLAG_NO_RANDSTROBES : 0));
        b.nam_cnt[r] = total;
        b.hit_total[r] = 0;
        b.rhit_total[r] = 0;
    }
    wave_sync_mem();
}

// The merge of up to four stashed reads (read k's hits in stash[k] for
// k < 3, the fourth read's in slot3) on one wave, 16 lanes a read, as
// k_merge4 merges them. A read a strand of which needs more than 16 NAMs is
// then merged alone from its stash, and spilled if its NAMs exceed F_NAMCAP.
// meta: the reads' ids (0..3), hit counts (4..7) and forward hits (8..11), in
// LDS.
__device__ __forceinline__ void fused_quad_merge(const DevBatch &b, DevHit (*stash)[64], DevHit *slot3, uint32_t qn,
                                                 const uint32_t *meta) {
    const uint32_t lane = lane_id(), seg = lane / SEG, j = lane % SEG;
    const bool act = seg < qn;
    const uint32_t r = meta[seg], nh = act ? meta[4 + seg] : 0u, nf = act ? meta[8 + seg] : 0u;
    const DevHit *mine = seg < 3 ? stash[seg] : slot3;
    const uint32_t total = merge_segments(mine, nh, nf, b.nam_slots + (uint64_t)r * F_NAMCAP);
    if (act && j == 0 && total != MERGE_OVERFLOW) b.nam_cnt[r] = total;
    uint64_t redo = ballot(act && j == 0 && total == MERGE_OVERFLOW);
    wave_sync_mem();
    while (redo) {
        const uint32_t l = (uint32_t)__builtin_ctzll(redo);
        redo &= redo - 1;
        const uint32_t rk = readlane_u32(r, l), nk = readlane_u32(nh, l);
        const uint32_t all = merge_arrival(l / SEG < 3 ? stash[l / SEG] : slot3, nk,
                                           b.nam_slots + (uint64_t)rk * F_NAMCAP, (uint32_t)F_NAMCAP);
        if (all > (uint32_t)F_NAMCAP) {
            spill_read(b, rk);
        } else {
            if (lane == 0) b.nam_cnt[rk] = all;
            wave_sync_mem();
        }
    }
}

// Six waves per SIMD: at most 80 VGPRs, and LDS for six 4-wave blocks per
// CU. A wave merges its reads four at a time (fused_quad_merge) once their
// hits wait in its stash: three slots in the stash, and the fourth read's
// hits left in the wave's own merge area, which nothing else touches until
// the four-read merge has run (the next read's seeding comes after it).
template <int LMAX, int FWPB, bool K20>
__global__ __launch_bounds__(64 * FWPB) __attribute__((amdgpu_waves_per_eu(6))) void k_fused(
    DevBatch b, DevIndex ix, SeedParams P, uint32_t rescue_cutoff, uint32_t hard_cutoff,
    const uint32_t *__restrict__ queue, uint32_t count, uint32_t chunk, unsigned int *head) {
    if (K20) pin_k20_profile(P);
    __shared__ FusedLds<LMAX> lds[FWPB];
    __shared__ DevHit qstash[FWPB][3][64];
    __shared__ uint32_t qmeta[FWPB][12];
    const int wid = (int)uni32(threadIdx.x >> 6);
    FusedLds<LMAX> &S = lds[wid];
    DevHit(*stash)[64] = qstash[wid];
    uint32_t *meta = qmeta[wid];
    uint32_t qn = 0;
    // a grid with a wave per read merges each read alone
    const bool alone = chunk == 0 && (uint64_t)gridDim.x * FWPB >= count;
    // static: queue entries w, w + W, ...; dynamic: grabs of `chunk` entries,
    // and every wave leaves once a grab starts at or past the end
    uint32_t w = chunk == 0 ? wave_index(FWPB) : 0u, end = 0;
    for (;;) {
        bool have;
        if (chunk == 0) {
            have = w < count;
        } else {
            if (w >= end) {
                uint32_t start = 0;
                if (lane_id() == 0) start = atomicAdd(head, chunk);
                start = (uint32_t)__builtin_amdgcn_readfirstlane((int)start);
                w = start;
                end = count - min(start, count) < chunk ? count : start + chunk;
            }
            have = w < end;
        }
        if (have) {
            const uint32_t r = sload(queue + w);
            w += chunk == 0 ? gridDim.x * FWPB : 1u;
            uint32_t nh = 0, nf = 0;
            DevHit *slot = qn < 3 ? stash[qn] : S.merge.hits;
            fused_read<LMAX>(b, ix, P, S, r, rescue_cutoff, hard_cutoff, alone ? nullptr : slot, nh, nf);
            if (nh) {
                if (lane_id() == 0) {
                    meta[qn] = r;
                    meta[4 + qn] = nh;
                    meta[8 + qn] = nf;
                }
                wave_sync_mem();
                qn++;
            }
        }
        if (qn == 4 || (!have && qn)) {
            fused_quad_merge(b, stash, S.merge.hits, qn, meta);
            qn = 0;
        }
        if (!have) break;
    }
}

// ---------------------------------------------------------------------------
// dense output: NAMs of read r to nams_out[nam_off[r] ..]

constexpr int SCAN_BLOCK = 256, SCAN_ITEMS = 4, SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;
constexpr uint32_t COMPACT_SEG = 16;
constexpr uint32_t COMPACT_SEG_WORDS = 8 * COMPACT_SEG;  // 11 NAMs of 11 words

// the control block with its totals to the host's copy, by the first thread
__device__ __forceinline__ void ctl_store(const DevBatch &b, DevCtl *dst, uint64_t nams, unsigned overflow) {
    if (threadIdx.x == 0) {
        DevCtl c = *b.ctl;
        c.overflow |= overflow;
        c.tot[0] = (uint64_t)b.n_reads * HIT_REGION + c.hit_pool;
        c.tot[1] = c.rhit_pool;
        c.tot[2] = nams;
        *dst = c;
    }
}

// sum of a[0 .. n) over the wave
__device__ __forceinline__ uint64_t wave_sum_of(const uint64_t *a, uint32_t n) {
    uint64_t v = 0;
    for (uint32_t t = lane_id(); t < n; t += 64) v += a[t];
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

// NAM offsets and the dense output. nam_off holds each read's offset inside its
// tile of SCAN_TILE reads and tiles the tiles' NAM counts (k_scan_tiles); each
// wave adds the counts of the tiles before its reads' own (ntiles > 0), or
// takes their prefix (ntiles == 0: tiles holds it, nam_off[n] the total). The
// first block hands the totals to the host.
__global__ __launch_bounds__(64 * WPB) void k_compact(DevBatch b, int fused, const uint64_t *tiles, uint32_t ntiles,
                                                      DevCtl *dst) {
    const uint32_t lane = lane_id();
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        const uint64_t total = ntiles ? wave_sum_of(tiles, ntiles) : b.nam_off[b.n_reads];
        if (lane == 0) {
            b.nam_off[b.n_reads] = total;
            if (b.h_off) b.h_off[b.n_reads] = total;
        }
        ctl_store(b, dst, total, total > b.out_cap ? (unsigned)OVF_OUT : 0u);
    }
    // the merges did not run and the counts are stale
    if (hits_missing(b)) return;
    // COMPACT_SEG lanes per read, so that a wave's reads start their loads
    // (count, flags, offsets, then NAMs) together; reads with more than
    // COMPACT_SEG_WORDS words of NAMs (repeats) are copied by the whole wave
    // afterwards, four words per lane in flight
    const uint32_t seg = lane / COMPACT_SEG, j = lane % COMPACT_SEG;
    const uint32_t per_wave = 64 / COMPACT_SEG;
    const uint32_t r0 = wave_index(WPB) * per_wave;
    if (r0 < b.n_reads) {
        const uint32_t r = r0 + seg;
        // the read's count, flags and offsets load together (r clamped to a
        // valid read; lanes past the end copy nothing)
        const uint32_t rr = r < b.n_reads ? r : b.n_reads - 1;
        const uint32_t c0 = b.nam_cnt[rr];
        const uint8_t fl = b.flags[rr];
        const uint64_t ho = b.hit_off[rr], rho = b.rhit_off[rr], in_tile = b.nam_off[rr];
        // (a wave's reads lie in one tile)
        const uint32_t tile = r0 / SCAN_TILE;
        const uint64_t no = in_tile + (ntiles ? wave_sum_of(tiles, tile) : tiles[tile]);
        if (j == 0 && r < b.n_reads) {
            b.nam_off[r] = no;
            if (b.h_off) {
                b.h_off[r] = no;
                b.h_frac[r] = b.frac[r];
                b.h_flags[r] = fl;
            }
        }
        const uint32_t c = r < b.n_reads && no + c0 <= b.out_cap ? c0 : 0u;
        const gis_nam *srcn;
        if (fused && !(fl & FLAG_SPILL)) srcn = b.nam_slots + (uint64_t)rr * F_NAMCAP;
        else if (fl & GIS_FLAG_RESCUED) srcn = b.rnam_fin + rho;
        else srcn = b.nam_fin + ho;
        const uint32_t *src = reinterpret_cast<const uint32_t *>(srcn);
        uint32_t *dst = reinterpret_cast<uint32_t *>(b.nams_out + no);
        const uint32_t words = c * (uint32_t)(sizeof(gis_nam) / 4);
        const bool big = words > COMPACT_SEG_WORDS;
        if (!big && words > 0) {
            // every load issues before the first store (indices past the
            // read's words repeat its last word, and store nothing)
            uint32_t v[COMPACT_SEG_WORDS / COMPACT_SEG];
#pragma unroll
            for (uint32_t u = 0; u < COMPACT_SEG_WORDS / COMPACT_SEG; u++) {
                const uint32_t i = j + u * COMPACT_SEG;
                v[u] = src[i < words ? i : words - 1];
            }
#pragma unroll
            for (uint32_t u = 0; u < COMPACT_SEG_WORDS / COMPACT_SEG; u++) {
                const uint32_t i = j + u * COMPACT_SEG;
                if (i < words) dst[i] = v[u];
            }
        }
        uint64_t bigs = ballot(big && j == 0);
        while (bigs) {
            const uint32_t l = (uint32_t)__builtin_ctzll(bigs);
            bigs &= bigs - 1;
            const uint32_t wl = readlane_u32(words, l);
            const uint32_t *sl = reinterpret_cast<const uint32_t *>(
                (uint64_t)readlane_u32((uint32_t)(uintptr_t)src, l) |
                ((uint64_t)readlane_u32((uint32_t)((uintptr_t)src >> 32), l) << 32));
            uint32_t *dl = reinterpret_cast<uint32_t *>(
                (uint64_t)readlane_u32((uint32_t)(uintptr_t)dst, l) |
                ((uint64_t)readlane_u32((uint32_t)((uintptr_t)dst >> 32), l) << 32));
            // four loads in flight per lane before their stores
            uint32_t i = lane;
            for (; i + 192 < wl; i += 256) {
                const uint32_t v0 = sl[i], v1 = sl[i + 64], v2 = sl[i + 128], v3 = sl[i + 192];
                dl[i] = v0;
                dl[i + 64] = v1;
                dl[i + 128] = v2;
                dl[i + 192] = v3;
            }
            for (; i < wl; i += 64) dl[i] = sl[i];
        }
    }
}

__global__ void k_reset_ctl(DevCtl *ctl) { ctl_clear(ctl); }

// plain lookup over a list of hashes (the microbenchmark gpu_find,
// gpu_test.cu:186-215, with StrobemerIndex::find semantics)
// find (StrobemerIndex::find) of each hash through its bucket line
__global__ void k_find_flat(DevIndex ix, const uint64_t *hashes, uint64_t n, uint64_t *positions) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Probe p;
    p.key = hashes[i];
    probe_line(ix, p);
    if (probe_small(p)) {
        uint32_t lt, eq;
        probe_small_find(p, lt, eq);
    } else {
        p.pos = p.e - p.s < 0xffffffffull ? dev_find_in(ix, p.key, p.s, p.e, &p.scan) : dev_find(ix, p.key, &p.scan);
    }
    positions[i] = p.pos;
}

// ---------------------------------------------------------------------------
// exclusive scan u32 -> u64 offsets[n+1]

__device__ __forceinline__ uint64_t block_excl_scan_u64(uint64_t v, uint64_t *lds_w, uint64_t *total) {
    const uint32_t lane = lane_id(), wid = threadIdx.x >> 6;
    uint64_t x = v;
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t y = __shfl_up(x, d, 64);
        if (lane >= (uint32_t)d) x += y;
    }
    if (lane == 63) lds_w[wid] = x;
    __syncthreads();
    uint64_t off = 0, tot = 0;
    for (uint32_t w = 0; w < SCAN_BLOCK / 64; w++) {
        if (w < wid) off += lds_w[w];
        tot += lds_w[w];
    }
    __syncthreads();
    *total = tot;
    return off + x - v;
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_tiles(const uint32_t *in, uint64_t *out,
                                                           uint64_t n, uint64_t *tile_sums) {
    __shared__ uint64_t lw[SCAN_BLOCK / 64];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    uint64_t v[SCAN_ITEMS];
    uint64_t s = 0;
    for (int j = 0; j < SCAN_ITEMS; j++) {
        v[j] = base + j < n ? in[base + j] : 0;
        s += v[j];
    }
    uint64_t tot;
    uint64_t ex = block_excl_scan_u64(s, lw, &tot);
    for (int j = 0; j < SCAN_ITEMS; j++) {
        if (base + j < n) out[base + j] = ex;
        ex += v[j];
    }
    if (threadIdx.x == 0) {
        tile_sums[blockIdx.x] = tot;
        if (gridDim.x == 1) out[n] = tot;
    }
}

// single block: exclusive scan of the tile sums in place; out[n] = total
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_sums(uint64_t *tile_sums, uint64_t ntiles,
                                                          uint64_t *out, uint64_t n) {
    __shared__ uint64_t lw[SCAN_BLOCK / 64];
    uint64_t carry = 0;
    for (uint64_t t0 = 0; t0 < ntiles; t0 += SCAN_BLOCK) {
        const uint64_t t = t0 + threadIdx.x;
        const uint64_t v = t < ntiles ? tile_sums[t] : 0;
        uint64_t tot;
        const uint64_t ex = block_excl_scan_u64(v, lw, &tot);
        if (t < ntiles) tile_sums[t] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) out[n] = carry;
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_add(uint64_t *out, uint64_t n,
                                                         const uint64_t *tile_sums) {
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    const uint64_t add = tile_sums[blockIdx.x];
    for (int j = 0; j < SCAN_ITEMS; j++)
        if (base + j < n) out[base + j] += add;
}

// k_scan_sums and k_scan_add in one launch for up to SCAN_FEW_TILES tiles:
// each block adds the sums of the tiles before its own (one wave reads them),
// and the last block writes the total
constexpr unsigned SCAN_FEW_TILES = 256;

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_add_few(uint64_t *out, uint64_t n, const uint64_t *tile_sums,
                                                             uint32_t ntiles) {
    __shared__ uint64_t add_s;
    if (threadIdx.x < 64) {
        uint64_t v = 0;
        for (uint32_t t = threadIdx.x; t < blockIdx.x; t += 64) v += tile_sums[t];
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
        if (threadIdx.x == 0) {
            add_s = v;
            if (blockIdx.x == ntiles - 1) out[n] = v + tile_sums[blockIdx.x];
        }
    }
    __syncthreads();
    const uint64_t add = add_s;
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    for (int j = 0; j < SCAN_ITEMS; j++)
        if (base + j < n) out[base + j] += add;
}

// ---------------------------------------------------------------------------
// launch wrappers

static inline unsigned grid_for(uint64_t items, unsigned per_block) {
    return (unsigned)((items + per_block - 1) / per_block);
}

// blocks for a per-read kernel over a set: one wave per read for a full set,
// a bounded grid-stride grid for a spill list (its size is on the device):
// up to 2048 blocks, a whole GPU's worth of waves, since the fused kernel
// can hand on a few percent of a batch (repeat-rich reads with many NAMs),
// and a read's seeding or lookup is a chain of dependent steps
static inline unsigned grid_for_set(const DevBatch &b, const ReadSet &set, unsigned wpb) {
    const unsigned g = grid_for(b.n_reads, wpb);
    if (!set.ids) return g;
    return g < 2048u ? g : 2048u;
}

// blocks for a per-read kernel over a selected list (its length is on the
// device): enough waves to run every heavy read of the list at once
static inline unsigned grid_selected(const DevBatch &b) {
    const unsigned g = grid_for(b.n_reads, WPB);
    return g < 2048u ? (g ? g : 1u) : 2048u;
}

// The bucket lines (DevIndex::lines) from starts and the table, eight lanes a
// bucket: lane 0 writes the head, lane j > 0 record j - 1. Bound by the lines'
// own bytes (2^bits x 128): a wave's store covers eight whole lines, where one
// thread a bucket stored 16 bytes at a 128-byte stride (2^20 buckets: 38 us,
// before 142; 2^25: 1267 us, before 3931).
__global__ __launch_bounds__(256) void k_bucket_lines(const uint4 *rs, const uint64_t *starts, uint64_t nb,
                                                      uint4 *lines) {
    const uint32_t j = threadIdx.x % BUCKET_LINE;
    constexpr uint32_t PER_BLOCK = 256 / BUCKET_LINE;
    for (uint64_t bk = (uint64_t)blockIdx.x * PER_BLOCK + threadIdx.x / BUCKET_LINE; bk < nb;
         bk += (uint64_t)gridDim.x * PER_BLOCK) {
        const uint64_t s = starts[bk], size = starts[bk + 1] - s;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (j == 0)
            v = make_uint4((uint32_t)s, (uint32_t)(s >> 32), size < 0xffffffffull ? (uint32_t)size : 0xffffffffu, 0u);
        else if (j <= size)
            v = rs[s + j - 1];
        lines[bk * BUCKET_LINE + j] = v;
    }
}

void launch_bucket_lines(const uint4 *rs, const uint64_t *starts, int bits, uint4 *lines, hipStream_t st) {
    const uint64_t nb = 1ull << bits, g = nb * BUCKET_LINE / 256;
    hipLaunchKernelGGL(k_bucket_lines, dim3((unsigned)(g < 65536 ? g : 65536)), dim3(256), 0, st, rs, starts, nb, lines);
}

// Small arrays between pinned host memory and the device, read or written over PCIe
// by the kernel itself: the inputs of a small call from one pinned block, where
// seven hipMemcpyAsync of a few kilobytes cost 5-10 us each on the host and a blit
// kernel each on the device, and the small arrays of a large result back.
__global__ __launch_bounds__(256) void k_copy_in(CopyList c, DevCtl *ctl) {
    if (ctl && blockIdx.x == 0) ctl_clear(ctl);
    int i = 0;
    while (i + 1 < c.n && blockIdx.x >= c.block[i + 1]) i++;
    if (blockIdx.x >= c.block[c.n]) return;
    const uint32_t at = (blockIdx.x - c.block[i]) * CopyList::BLOCK_BYTES, bytes = c.bytes[i];
    const char *src = static_cast<const char *>(c.src[i]);
    char *dst = static_cast<char *>(c.dst[i]);
#pragma unroll
    for (uint32_t u = 0; u < CopyList::BLOCK_BYTES / 4096; u++) {
        const uint32_t o = at + u * 4096 + threadIdx.x * 16;
        if (o + 16 <= bytes) *reinterpret_cast<uint4 *>(dst + o) = *reinterpret_cast<const uint4 *>(src + o);
        else
            for (uint32_t k = o; k < bytes; k++) dst[k] = src[k];
    }
}

void launch_copy_in(const CopyList &c, DevCtl *ctl, hipStream_t st) {
    const unsigned g = c.block[c.n] ? c.block[c.n] : 1u;
    hipLaunchKernelGGL(k_copy_in, dim3(g), dim3(256), 0, st, c, ctl);
}

void launch_reset_ctl(DevCtl *ctl, hipStream_t st) {
    hipLaunchKernelGGL(k_reset_ctl, dim3(1), dim3(64), 0, st, ctl);
}

void launch_seed(const DevBatch &b, const ReadSet &set, const SeedParams &sp, int want_syncmers,
                 int long_reads, int reset, hipStream_t st) {
    if (b.n_reads == 0) {
        if (reset) launch_reset_ctl(b.ctl, st);
        return;
    }
    const unsigned g = grid_for_set(b, set, SEED_WPB);
    typedef void (*SeedKernel)(DevBatch, ReadSet, SeedParams, int, int);
    const bool k20 = is_k20_profile(sp);
    const SeedKernel short_k = k20 ? (SeedKernel)k_seed<false, true> : (SeedKernel)k_seed<false, false>;
    const SeedKernel long_k = k20 ? (SeedKernel)k_seed<true, true> : (SeedKernel)k_seed<true, false>;
    hipLaunchKernelGGL(short_k, dim3(g), dim3(64 * SEED_WPB), 0, st, b, set, sp, want_syncmers, reset);
    if (long_reads) hipLaunchKernelGGL(long_k, dim3(g * SEED_WPB), dim3(64), 0, st, b, set, sp, want_syncmers, 0);
}

void launch_emit_seeds(const DevBatch &b, int syncmers, const uint64_t *off, void *out, uint64_t *h_off,
                       hipStream_t st) {
    if (b.n_reads == 0) return;
    const unsigned g = grid_for(b.n_reads, WPB);
    hipLaunchKernelGGL(syncmers ? k_emit_syncmers : k_emit_randstrobes, dim3(g), dim3(64 * WPB), 0, st, b, off,
                       static_cast<uint64_t *>(out), h_off);
}

void launch_lookup(const DevBatch &b, const ReadSet &set, const DevIndex &ix, int rescue_mode,
                   hipStream_t st) {
    if (b.n_reads == 0) return;
    hipLaunchKernelGGL(k_lookup, dim3(grid_for_set(b, set, WPB)), dim3(64 * WPB), 0, st, b, set, ix,
                       rescue_mode, set.ids ? 1 : 0);
}

void launch_hits(const DevBatch &b, const DevIndex &ix, uint32_t rescue_cutoff, uint32_t hard_cutoff,
                 hipStream_t st) {
    if (b.n_reads == 0) return;
    hipLaunchKernelGGL(k_hits, dim3(grid_selected(b)), dim3(64 * WPB), 0, st, b, ix, rescue_cutoff, hard_cutoff);
}

// four reads per wave over the set, then the reads it handed on, one per wave,
// then the (strand, ref) groups of split reads and their finish
void launch_merge(const DevBatch &b, const ReadSet &set, hipStream_t st) {
    if (b.n_reads == 0) return;
    const unsigned g = grid_for_set(b, set, WPB);
    hipLaunchKernelGGL(k_merge4, dim3((g + RPW - 1) / RPW), dim3(64 * WPB), 0, st, b, set);
    hipLaunchKernelGGL(k_merge, dim3(grid_selected(b) * WPB), dim3(64), 0, st, b);
    if (b.merge_scratch) {
        hipLaunchKernelGGL(k_merge_groups, dim3(4096), dim3(64), 0, st, b);
        hipLaunchKernelGGL(k_merge_split_finish, dim3(256), dim3(64 * WPB), 0, st, b);
    }
}

// fused kernel over queue[0 .. count): FWPB waves per block, LMAX the LDS
// tiling (reads longer than LMAX spill), grid 0 = one wave per entry,
// chunk 0 = static round robin, else dynamic grabs of chunk entries.
template <int LMAX, int FWPB, bool K20>
static void launch_fused_t(const DevBatch &b, const DevIndex &ix, const SeedParams &sp, uint32_t rcut,
                           uint32_t hard, const uint32_t *queue, uint32_t count, unsigned grid,
                           uint32_t chunk, unsigned int *head, hipStream_t st) {
    const unsigned g1 = grid_for(count, FWPB);
    const unsigned g = grid == 0 || grid > g1 ? g1 : grid;
    hipLaunchKernelGGL((k_fused<LMAX, FWPB, K20>), dim3(g), dim3(64 * FWPB), 0, st, b, ix, sp, rcut, hard,
                       queue, count, chunk, head);
}

bool launch_fused(const DevBatch &b, const DevIndex &ix, const SeedParams &sp, uint32_t rcut,
                  uint32_t hard, const uint32_t *queue, uint32_t count, int lmax, int wpb, unsigned grid,
                  uint32_t chunk, unsigned int *head, hipStream_t st) {
    if (count == 0) return true;
#define GIS_FUSED_CASE(LM, W)                                                                      \
    if (lmax == LM && wpb == W) {                                                                  \
        if (is_k20_profile(sp))                                                                    \
            launch_fused_t<LM, W, true>(b, ix, sp, rcut, hard, queue, count, grid, chunk, head, st); \
        else                                                                                       \
            launch_fused_t<LM, W, false>(b, ix, sp, rcut, hard, queue, count, grid, chunk, head, st); \
        return true;                                                                               \
    }
    GIS_FUSED_CASE(160, 2) GIS_FUSED_CASE(160, 4) GIS_FUSED_CASE(160, 8)
    GIS_FUSED_CASE(320, 2) GIS_FUSED_CASE(320, 4) GIS_FUSED_CASE(320, 8)
#undef GIS_FUSED_CASE
    return false;
}

// n bytes of HBM to pinned memory, 16 a lane (both ends 16-byte aligned): a chunk
// of a large copy starts ~10 us sooner than on the copy engines
__global__ __launch_bounds__(256) void k_copy_out(const uint4 *__restrict__ src, uint4 *__restrict__ dst, uint64_t n) {
    const uint64_t whole = n / 16;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < whole; i += (uint64_t)gridDim.x * 256) dst[i] = src[i];
    const uint64_t t = whole * 16 + threadIdx.x;
    if (blockIdx.x == 0 && t < n) reinterpret_cast<uint8_t *>(dst)[t] = reinterpret_cast<const uint8_t *>(src)[t];
}

void launch_copy_out(const void *src, void *dst, uint64_t n, hipStream_t st) {
    const unsigned g = (unsigned)std::min<uint64_t>((n + 4095) / 4096, 512);
    hipLaunchKernelGGL(k_copy_out, dim3(g), dim3(256), 0, st, static_cast<const uint4 *>(src), static_cast<uint4 *>(dst), n);
}

// The control block to pinned host memory by a thread's stores, so that the
// end of a run takes no copy engine (the engines carry the batches' reads and
// NAMs).
__global__ void k_ctl_to_host(DevBatch b, DevCtl *dst) { ctl_store(b, dst, 0, 0u); }

void launch_ctl_to_host(const DevBatch &b, DevCtl *dst, hipStream_t st) {
    hipLaunchKernelGGL(k_ctl_to_host, dim3(1), dim3(64), 0, st, b, dst);
}

// Up to SCAN_OWN_TILES tiles each wave of k_compact sums the tiles before its
// own (a load a lane for 64 tiles), which saves the launch that would turn them
// into a prefix; beyond (1,048,576 reads) that launch is the cheaper way.
constexpr unsigned SCAN_OWN_TILES = 1024;

void launch_output(const DevBatch &b, int fused, uint64_t *tmp, DevCtl *dst, hipStream_t st) {
    const uint64_t n = b.n_reads;
    if (n == 0) {
        launch_scan(b.nam_cnt, b.nam_off, 0, tmp, st);
        launch_ctl_to_host(b, dst, st);
        return;
    }
    unsigned tiles = grid_for(n, SCAN_TILE);
    hipLaunchKernelGGL(k_scan_tiles, dim3(tiles), dim3(SCAN_BLOCK), 0, st, b.nam_cnt, b.nam_off, n, tmp);
    if (tiles > SCAN_OWN_TILES) {
        hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_BLOCK), 0, st, tmp, (uint64_t)tiles, b.nam_off, n);
        tiles = 0;
    }
    hipLaunchKernelGGL(k_compact, dim3(grid_for(n, WPB * (64 / COMPACT_SEG))), dim3(64 * WPB), 0, st, b, fused, tmp,
                       (uint32_t)tiles, dst);
}

void launch_find_flat(const DevIndex &ix, const uint64_t *hashes, uint64_t n, uint64_t *positions,
                      hipStream_t st) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_find_flat, dim3(grid_for(n, 256)), dim3(256), 0, st, ix, hashes, n, positions);
}

size_t scan_tmp_words(uint64_t n) { return (size_t)grid_for(n ? n : 1, SCAN_TILE) + 1; }

void launch_scan(const uint32_t *in, uint64_t *out, uint64_t n, uint64_t *tmp, hipStream_t st) {
    const unsigned tiles = grid_for(n ? n : 1, SCAN_TILE);
    if (n > 0 && tiles <= SCAN_FEW_TILES) {
        hipLaunchKernelGGL(k_scan_tiles, dim3(tiles), dim3(SCAN_BLOCK), 0, st, in, out, n, tmp);
        if (tiles == 1) return;
        hipLaunchKernelGGL(k_scan_add_few, dim3(tiles), dim3(SCAN_BLOCK), 0, st, out, n, tmp, (uint32_t)tiles);
        return;
    }
    if (n > 0)
        hipLaunchKernelGGL(k_scan_tiles, dim3(tiles), dim3(SCAN_BLOCK), 0, st, in, out, n, tmp);
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_BLOCK), 0, st, tmp, (uint64_t)(n ? tiles : 0), out, n);
    if (n > 0) hipLaunchKernelGGL(k_scan_add, dim3(tiles), dim3(SCAN_BLOCK), 0, st, out, n, tmp);
}

}  // namespace gis
