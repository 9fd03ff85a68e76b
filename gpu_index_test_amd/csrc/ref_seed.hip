// Device seeding of the reference for the index build: the RefRandstrobe
// records of every contig, as the reference's RandstrobeGenerator makes
// them over each contig's syncmers (step2/randstrobes.cu:18-79,136-190;
// count/assign_randstrobes at step2/index.cu:246-311).
//
// The contigs sit in HBM back to back with one 'N' after each, so a contig
// boundary acts as an N run: no window spans two contigs and the first
// window after a boundary starts a segment. The scan runs as passes over
// the whole genome, each a grid over positions:
//   1. bases packed 2 bits each, with a mask of non-ACGT bases, sixteen a lane;
//   2. a tile of k-mer windows a block: the canonical s-mer hashes in LDS, and
//      from them the state of every window that needs no history (segment
//      starts and windows with a unique minimum below ~0, gis_core.h);
//   3. each maximal run of windows with tied minima replayed from the known
//      window before it by one lane (slide, gis_core.h), its hashes computed
//      again -- tied runs are rare and short except in tandem repeats, and a
//      run's replay is sequential in the reference too;
//   4. syncmer positions compacted per 4096-window tile (scan of tile
//      counts), then the canonical k-mer hash of each syncmer;
//   5. per contig, the range of its syncmers; then one lane per syncmer
//      picks its partner among the next w_min..w_max syncmers of the contig
//      within max_dist (the smallest popcount((h_i ^ h_j) & q), earliest on
//      ties) and writes its record. A contig's last w_min syncmers start no
//      randstrobe; a contig shorter than w_max gets zero records in its
//      slots, as the reference counts them but never assigns them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "index_build.h"
#include "kernels.h"
#include "seed_dev.h"
#include "wave.h"

namespace gis {

namespace {

constexpr int TILE_THREADS = 256, TILE_WIN = 16, TILE = TILE_THREADS * TILE_WIN;

void check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw BuildError{e, what};
}

unsigned grid(uint64_t items, unsigned per_block) {
    const uint64_t g = (items + per_block - 1) / per_block;
    return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(g, 1u << 20));
}

#define GRID_STRIDE(i, n) \
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (uint64_t)gridDim.x * blockDim.x)

// 1. sixteen bases a lane: a 32-bit word of packed bases and 16 bits of the N
// mask; past the end reads as N
__global__ __launch_bounds__(256) void k_ref_pack(const uint4 *__restrict__ seq, uint64_t T, uint64_t n16,
                                                  uint32_t *__restrict__ pk, uint16_t *__restrict__ nmask) {
    GRID_STRIDE(w, n16) {
        const uint64_t first = 16 * w;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (first < T) v = seq[w];  // (the array is padded to 16 bytes)
        const uint32_t in[4] = {v.x, v.y, v.z, v.w};
        uint32_t p = 0, n = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            uint32_t bad;
            p |= pack4(nt4x4(in[u], bad)) << (8 * u);
#pragma unroll
            for (int q = 0; q < 4; q++) n |= (bad >> (8 * q) & 0xffu) != 0 ? 1u << (4 * u + q) : 0u;
        }
        if (first + 16 > T) n |= first >= T ? 0xffffu : 0xffffu << (T - first) & 0xffffu;
        pk[w] = p;
        nmask[w] = (uint16_t)n;
    }
}

// the 'N' after each contig
__global__ void k_ref_separators(char *__restrict__ seq, const uint64_t *__restrict__ cstart, uint32_t n_refs) {
    GRID_STRIDE(c, n_refs) seq[cstart[c + 1] - 1] = 'N';
}

// canonical s-mer hash at base j
__device__ __forceinline__ uint64_t smer_hash(const uint64_t *pk, uint64_t j, const SeedParams &P) {
    return xxh64_u64(canonical_code(pk, j, P.s, P.smask));
}

// 2. window states that need no history, WIN windows a block. The s-mer hashes
// stay in LDS, high words apart: they decide a window unless two of them tie.
// The hashes' 64-bit products bound it. (20.0 M windows: 77 us; a pass that wrote
// the hashes and one that read five of them a window took 88 us each and 160 MB.)
// S16: s <= 16, an s-mer's code is one 32-bit word.
constexpr int WIN = 2048, WIN_MAX_W = 32;

template <bool S16>
__global__ __launch_bounds__(256) void k_ref_windows(const uint64_t *__restrict__ pk,
                                                     const uint64_t *__restrict__ nmask, uint64_t ns, uint64_t nk,
                                                     SeedParams P, uint8_t *__restrict__ st) {
    __shared__ uint32_t hi[WIN + WIN_MAX_W], lo[WIN + WIN_MAX_W];
    const uint64_t p0 = (uint64_t)blockIdx.x * WIN;
    const uint64_t *bpk = pk + p0 / 32;
    const int bns = ns > p0 ? (int)std::min<uint64_t>(ns - p0, WIN + WIN_MAX_W) : 0;
    // (s-mers with a non-ACGT base lie in invalid windows only)
    for (int i = threadIdx.x; i < WIN + P.w - 1; i += 256) {
        uint64_t h = 0;
        if (i < bns)
            h = xxh64_u64(S16 ? canonical_code32(bpk, i, P.s, (uint32_t)P.smask)
                              : canonical_code(bpk, i, P.s, P.smask));
        hi[i] = (uint32_t)(h >> 32);
        lo[i] = (uint32_t)h;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < WIN; i += 256) {
        const uint64_t p = p0 + i;
        if (p >= nk) break;
        uint8_t s;
        if (any_n(nmask, p, p + (uint64_t)P.k - 1)) {
            s = ST_INVALID;
        } else {
            uint32_t m = hi[i];
            int at = 0, eq = 1;
            for (int o = 1; o < P.w; o++) {
                const uint32_t v = hi[i + o];
                eq = v < m ? 1 : eq + (v == m ? 1 : 0);
                at = v < m ? o : at;
                m = min(m, v);
            }
            s = (uint8_t)at;
            if (eq > 1) {  // the full hashes decide
                uint64_t mv = UINT64_MAX;
                int first = 0, ties = 0;
                for (int o = 0; o < P.w; o++) {
                    const uint64_t v = ((uint64_t)hi[i + o] << 32) | lo[i + o];
                    if (v < mv) { mv = v; first = o; ties = 1; }
                    else if (v == mv) ties++;
                }
                const bool seg_first = p == 0 || ((nmask[(p - 1) >> 6] >> ((p - 1) & 63)) & 1);
                if (seg_first) s = mv == UINT64_MAX ? ST_NONE : (uint8_t)first;
                else s = ties == 1 && mv != UINT64_MAX ? (uint8_t)first : ST_UNKNOWN;
            } else if (m == 0xffffffffu && lo[i + at] == 0xffffffffu) {
                // a minimum of ~0 (one window of one s-mer)
                const bool seg_first = p == 0 || ((nmask[(p - 1) >> 6] >> ((p - 1) & 63)) & 1);
                s = seg_first ? ST_NONE : ST_UNKNOWN;
            }
        }
        st[p] = s;
    }
}

// 3. each run of tied windows replayed from the known window before it (a
// run never starts a segment: a segment's first window is an anchor). The
// resolved states go to st2, so that st, which decides where runs start,
// never changes under the other lanes.
__global__ void k_ref_resolve(const uint64_t *__restrict__ pk,
                              const uint8_t *__restrict__ st, uint64_t nk, SeedParams P,
                              uint8_t *__restrict__ st2) {
    // sixteen windows a lane: unknown ones are rare
    GRID_STRIDE(g, (nk + 15) / 16) {
        const uint4 v = reinterpret_cast<const uint4 *>(st)[g];  // (padded)
        const uint32_t u4 = 0x01010101u * ST_UNKNOWN, w[4] = {v.x ^ u4, v.y ^ u4, v.z ^ u4, v.w ^ u4};
        bool any = false;
#pragma unroll
        for (int q = 0; q < 4; q++) any |= ((w[q] - 0x01010101u) & ~w[q] & 0x80808080u) != 0;
        if (!any) continue;
        for (uint64_t p = std::max<uint64_t>(16 * g, 1); p < std::min(16 * g + 16, nk); p++) {
            if (st[p] != ST_UNKNOWN || st[p - 1] == ST_UNKNOWN) continue;
            // slide (gis_core.h) with the tracked hash kept; no base of these
            // windows is an N
            uint8_t r = st[p - 1];
            uint64_t tracked = r == ST_NONE ? UINT64_MAX : smer_hash(pk, p - 1 + r, P);
            for (uint64_t x = p; x < nk && st[x] == ST_UNKNOWN; x++) {
                const uint64_t v = smer_hash(pk, x + P.w - 1, P);
                if (r == 0) {  // left the window: its rightmost minimum
                    r = (uint8_t)(P.w - 1);
                    tracked = v;
                    for (int o = P.w - 2; o >= 0; o--) {
                        const uint64_t c = smer_hash(pk, x + o, P);
                        if (c < tracked) { tracked = c; r = (uint8_t)o; }
                    }
                } else if (v < tracked) {
                    r = (uint8_t)(P.w - 1);
                    tracked = v;
                } else if (r != ST_NONE) {
                    r--;
                }
                st2[x] = r;
            }
        }
    }
}

// which of the TILE_WIN windows from base on (a multiple of it) are syncmers
static_assert(TILE_WIN == 16, "one 16-byte load of states");
__device__ __forceinline__ uint32_t sync_flags(const uint8_t *st, const uint8_t *st2, uint64_t base, uint64_t nk,
                                               int t) {
    if (base >= nk) return 0;
    const uint4 v = *reinterpret_cast<const uint4 *>(st + base);  // (padded)
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    const uint32_t want = (uint32_t)(t - 1);
    uint32_t f = 0, unknown = 0;
#pragma unroll
    for (int u = 0; u < TILE_WIN; u++) {
        const uint32_t s = w[u / 4] >> (8 * (u % 4)) & 0xffu;
        f |= s == want ? 1u << u : 0u;
        unknown |= s == ST_UNKNOWN ? 1u << u : 0u;
    }
    if (base + TILE_WIN > nk) {
        const uint32_t in = (1u << (nk - base)) - 1u;
        f &= in;
        unknown &= in;
    }
    while (unknown) {
        const uint32_t u = (uint32_t)__builtin_ctz(unknown);
        unknown &= unknown - 1;
        if (st2[base + u] == (uint8_t)want) f |= 1u << u;
    }
    return f;
}

// 4a. syncmers per tile of TILE windows
__global__ __launch_bounds__(TILE_THREADS) void k_ref_sync_count(const uint8_t *__restrict__ st,
                                                                 const uint8_t *__restrict__ st2, uint64_t nk,
                                                                 int t, uint32_t *__restrict__ cnt) {
    __shared__ uint32_t part[TILE_THREADS / 64];
    const uint64_t base = (uint64_t)blockIdx.x * TILE + (uint64_t)threadIdx.x * TILE_WIN;
    const uint32_t c = wave_sum((uint32_t)__popc(sync_flags(st, st2, base, nk, t)));
    if (lane_id() == 0) part[threadIdx.x / 64] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = 0;
        for (int i = 0; i < TILE_THREADS / 64; i++) s += part[i];
        cnt[blockIdx.x] = s;
    }
}

// 4b. syncmer positions in order: tile offset + rank inside the tile
__global__ __launch_bounds__(TILE_THREADS) void k_ref_sync_write(const uint8_t *__restrict__ st,
                                                                 const uint8_t *__restrict__ st2, uint64_t nk,
                                                                 int t, const uint64_t *__restrict__ tile_off,
                                                                 uint64_t *__restrict__ sy_pos) {
    __shared__ uint32_t part[TILE_THREADS / 64];
    const uint64_t base = (uint64_t)blockIdx.x * TILE + (uint64_t)threadIdx.x * TILE_WIN;
    const uint32_t flags = sync_flags(st, st2, base, nk, t), c = (uint32_t)__popc(flags);
    const uint32_t ex = wave_excl_scan(c);
    const uint32_t wtot = wave_sum(c);
    const uint32_t wid = threadIdx.x / 64;
    if (lane_id() == 0) part[wid] = wtot;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t i = 0; i < wid; i++) before += part[i];
    uint64_t at = tile_off[blockIdx.x] + before + ex;
    for (int u = 0; u < TILE_WIN; u++)
        if ((flags >> u) & 1u) sy_pos[at++] = base + u;
}

// 4c. canonical k-mer hash of each syncmer
__global__ void k_ref_sync_hash(const uint64_t *__restrict__ pk, const uint64_t *__restrict__ sy_pos, uint64_t n,
                                SeedParams P, uint64_t *__restrict__ sy_hash) {
    GRID_STRIDE(i, n) sy_hash[i] = xxh64_u64(canonical_code(pk, sy_pos[i], P.k, P.kmask));
}

// 5a. first syncmer of each contig (and n at the end): lower bound of the
// contig's first base among the syncmer positions
__global__ void k_ref_contig_syncmers(const uint64_t *__restrict__ sy_pos, uint64_t n,
                                      const uint64_t *__restrict__ cstart, uint32_t n_refs,
                                      uint64_t *__restrict__ sy_start) {
    GRID_STRIDE(c, (uint64_t)n_refs + 1) {
        const uint64_t key = cstart[c];
        uint64_t lo = 0, cnt = n;
        while (cnt > 0) {
            const uint64_t step = cnt >> 1, it = lo + step;
            if (sy_pos[it] < key) {
                lo = it + 1;
                cnt -= step + 1;
            } else {
                cnt = step;
            }
        }
        sy_start[c] = c == n_refs ? n : lo;
    }
}

// 5b. the randstrobe of each syncmer that starts one
__global__ void k_ref_randstrobes(const uint64_t *__restrict__ sy_pos, const uint64_t *__restrict__ sy_hash,
                                  uint64_t n, const uint64_t *__restrict__ sy_start,
                                  const uint64_t *__restrict__ rs_start, const uint64_t *__restrict__ cstart,
                                  const uint8_t *__restrict__ is_short, uint32_t n_refs, SeedParams P,
                                  uint4 *__restrict__ out, uint64_t *__restrict__ o_hash,
                                  uint64_t *__restrict__ o_sec) {
    GRID_STRIDE(i, n) {
        // the contig: last c with sy_start[c] <= i
        uint32_t lo = 0, hi = n_refs;  // sy_start[lo] <= i < sy_start[hi]
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (sy_start[mid] <= i) lo = mid;
            else hi = mid;
        }
        while (lo + 1 < n_refs && sy_start[lo + 1] <= i) lo++;
        const uint32_t c = lo;
        const uint64_t first = sy_start[c], last = sy_start[c + 1] - 1;  // the contig's syncmers
        if (i + P.w_min > last) continue;  // fewer than w_min syncmers follow
        const uint64_t o = rs_start[c] + (i - first);
        if (is_short[c]) {
            if (out) out[o] = make_uint4(0u, 0u, 0u, 0u);
            else o_hash[o] = o_sec[o] = 0;
            continue;
        }
        const uint64_t hi_ = sy_hash[i], pi = sy_pos[i];
        const uint64_t wend = std::min<uint64_t>(i + P.w_max, last);
        const uint64_t maxp = pi + P.max_dist_u;
        uint64_t best = i, bh = hi_;
        uint32_t minv = 0xffffffffu;
        for (uint64_t j = i + P.w_min; j <= wend; j++) {
            const uint64_t pj = sy_pos[j];
            if (pj > maxp) break;
            const uint64_t hj = sy_hash[j];
            const uint32_t cnt = (uint32_t)__popcll((hi_ ^ hj) & P.q);
            if (cnt < minv) {
                minv = cnt;
                best = j;
                bh = hj;
            }
        }
        const uint64_t hash = hi_ + bh;
        const uint32_t pos = (uint32_t)(pi - cstart[c]);
        const uint32_t packed = (c << 8) + (uint32_t)(sy_pos[best] - pi);
        if (out) {
            out[o] = make_uint4((uint32_t)hash, (uint32_t)(hash >> 32), pos, packed);
        } else {
            o_hash[o] = hash;
            o_sec[o] = ((uint64_t)pos << 32) | packed;
        }
    }
}

}  // namespace

RefSeeds device_seed_reference(const char *const *seqs, const uint64_t *lens, uint32_t n_refs, const gis_params &gp,
                               bool split, BuildArena &arena, hipStream_t st) {
    RefSeeds out;
    const SeedParams P = make_seed_params(gp);
    // contig c at cstart[c], one 'N' after each; cstart[n_refs] = T
    std::vector<uint64_t> cstart(n_refs + 1), sy_start(n_refs + 1), rs_start(n_refs + 1);
    std::vector<uint8_t> is_short(std::max<uint32_t>(n_refs, 1), 0);
    uint64_t T = 0, longest = 0;
    for (uint32_t c = 0; c < n_refs; c++) {
        cstart[c] = T;
        T += lens[c] + 1;
        longest = std::max(longest, lens[c]);
    }
    cstart[n_refs] = T;
    // (all host arrays here outlive the copies: the stream is waited for before
    // they go, also on the way out of an error)
    struct Drain {
        hipStream_t st;
        ~Drain() { (void)hipStreamSynchronize(st); }
    } drain{st};
    const uint64_t nwords = (T + 63) / 64;
    char *seq = arena.get<char>(T + 16);
    uint64_t *cs = arena.get<uint64_t>(n_refs + 1);
    check(hipMemcpyAsync(cs, cstart.data(), 8ull * (n_refs + 1), hipMemcpyHostToDevice, st), "contig starts");
    for (uint32_t c = 0; c < n_refs; c++)
        if (lens[c])
            check(hipMemcpyAsync(seq + cstart[c], seqs[c], lens[c], hipMemcpyHostToDevice, st), "genome upload");
    hipLaunchKernelGGL(k_ref_separators, dim3(grid(n_refs, 256)), dim3(256), 0, st, seq, cs, n_refs);
    // pad words: canonical_code reads the word after a window's first, any_n the
    // last one's
    uint64_t *pk = arena.get<uint64_t>(2 * nwords + 2);
    uint64_t *nm = arena.get<uint64_t>(nwords + 1);
    const uint64_t n16 = 4 * nwords + 4;
    hipLaunchKernelGGL(k_ref_pack, dim3(grid(n16, 256)), dim3(256), 0, st, reinterpret_cast<const uint4 *>(seq), T,
                       n16, reinterpret_cast<uint32_t *>(pk), reinterpret_cast<uint16_t *>(nm));
    check(hipGetLastError(), "k_ref_pack");

    const uint64_t ns = T >= (uint64_t)P.s ? T - P.s + 1 : 0;
    const uint64_t nk = T >= (uint64_t)P.k ? T - P.k + 1 : 0;
    if (nk == 0) return out;
    if (P.w > WIN_MAX_W) throw BuildError{hipErrorInvalidValue, "windows of more than 32 s-mers"};
    uint8_t *stt = arena.get<uint8_t>(nk + 16);
    uint8_t *st2 = arena.get<uint8_t>(nk + 16);
    hipLaunchKernelGGL(P.s <= 16 ? k_ref_windows<true> : k_ref_windows<false>, dim3((unsigned)((nk + WIN - 1) / WIN)), dim3(256), 0, st, pk, nm, ns, nk, P,
                       stt);
    check(hipGetLastError(), "k_ref_windows");
    hipLaunchKernelGGL(k_ref_resolve, dim3(grid((nk + 15) / 16, 256)), dim3(256), 0, st, pk, stt, nk, P, st2);
    check(hipGetLastError(), "k_ref_resolve");

    const uint64_t ntiles = (nk + TILE - 1) / TILE;
    uint32_t *cnt = arena.get<uint32_t>(ntiles);
    uint64_t *toff = arena.get<uint64_t>(ntiles + 1);
    uint64_t *tmp = arena.get<uint64_t>(scan_tmp_words(ntiles) + 8);
    hipLaunchKernelGGL(k_ref_sync_count, dim3((unsigned)ntiles), dim3(TILE_THREADS), 0, st, stt, st2, nk, P.t, cnt);
    check(hipGetLastError(), "k_ref_sync_count");
    launch_scan(cnt, toff, ntiles, tmp, st);
    check(hipGetLastError(), "syncmer scan");
    uint64_t nsy = 0;
    check(hipMemcpyAsync(&nsy, toff + ntiles, 8, hipMemcpyDeviceToHost, st), "syncmer count");
    check(hipStreamSynchronize(st), "syncmer count");
    uint64_t *pos = arena.get<uint64_t>(nsy);
    hipLaunchKernelGGL(k_ref_sync_write, dim3((unsigned)ntiles), dim3(TILE_THREADS), 0, st, stt, st2, nk, P.t, toff,
                       pos);
    check(hipGetLastError(), "k_ref_sync_write");
    uint64_t *hsh = arena.get<uint64_t>(nsy);
    hipLaunchKernelGGL(k_ref_sync_hash, dim3(grid(nsy, 256)), dim3(256), 0, st, pk, pos, nsy, P, hsh);
    check(hipGetLastError(), "k_ref_sync_hash");

    // per contig: syncmer range, randstrobe slots, short contigs
    uint64_t *sys = arena.get<uint64_t>(n_refs + 1);
    hipLaunchKernelGGL(k_ref_contig_syncmers, dim3(grid(n_refs + 1, 256)), dim3(256), 0, st, pos, nsy, cs, n_refs,
                       sys);
    check(hipGetLastError(), "k_ref_contig_syncmers");
    check(hipMemcpyAsync(sy_start.data(), sys, 8ull * (n_refs + 1), hipMemcpyDeviceToHost, st), "syncmer ranges");
    check(hipStreamSynchronize(st), "syncmer ranges");
    uint64_t total = 0;
    for (uint32_t c = 0; c < n_refs; c++) {
        rs_start[c] = total;
        const uint64_t nc = sy_start[c + 1] - sy_start[c];
        const uint64_t nr = nc > gp.w_min ? nc - gp.w_min : 0;
        total += nr;
        is_short[c] = lens[c] < gp.w_max ? 1 : 0;
        out.zeros |= is_short[c] && nr > 0;
    }
    rs_start[n_refs] = total;
    uint64_t *rss = arena.get<uint64_t>(n_refs + 1);
    uint8_t *shrt = arena.get<uint8_t>(n_refs);
    check(hipMemcpyAsync(rss, rs_start.data(), 8ull * (n_refs + 1), hipMemcpyHostToDevice, st), "slot starts");
    check(hipMemcpyAsync(shrt, is_short.data(), n_refs, hipMemcpyHostToDevice, st), "short contigs");
    out.n = total;
    // one contig's positions ascend
    out.pos_bits = n_refs > 1 && longest > 1 ? 64 - __builtin_clzll(longest - 1) : 0;
    if (split) {
        out.hash = arena.get<uint64_t>(total);
        out.sec = arena.get<uint64_t>(total);
    } else {
        out.recs = arena.get<uint4>(total);
    }
    hipLaunchKernelGGL(k_ref_randstrobes, dim3(grid(nsy, 256)), dim3(256), 0, st, pos, hsh, nsy, sys, rss, cs, shrt,
                       n_refs, P, out.recs, out.hash, out.sec);
    check(hipGetLastError(), "k_ref_randstrobes");
    check(hipStreamSynchronize(st), "k_ref_randstrobes");
    return out;
}

}  // namespace gis
