// Device half of strobemer index construction (StrobemerIndex::populate,
// step2/index.cu:143-244): sort the RefRandstrobe records by (hash,
// position, packed), fill the bucket starts with the reference's rule for
// where a bucket begins, and histogram the runs of equal hashes.
//
// Up to MAX_PARTS x PART_MEAN records (about 80 Mbp of reference) the sort is one
// partition by the top hash bits, into parts that fit a block's LDS, and a sort of
// each part there: the records are read and written three times in all (4.0 M
// records: 121 us, where the digit passes of the library took 640 us). Beyond that, or
// where a part overflows (a hash held by thousands of records), it is two stable
// LSD radix sorts of the library (rocPRIM): first by position, then by hash. The
// records come in contig order, so equal (hash, position) stay in the order of
// their packed word without sorting by it, and a single contig's positions ascend
// already. The bucket starts and the histogram are plain grid-stride kernels over
// the sorted table.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>

#include "index_build.h"
#include "kernels.h"
#include "wave.h"

namespace gis {

namespace {

__global__ void k_pack(uint4 *__restrict__ rs, uint64_t n, const uint64_t *__restrict__ hash,
                       const uint64_t *__restrict__ sec) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t h = hash[i], p = sec[i];
        rs[i] = make_uint4((uint32_t)h, (uint32_t)(h >> 32), (uint32_t)(p >> 32), (uint32_t)p);
    }
}

__global__ void k_fill(uint64_t *__restrict__ a, uint64_t n, uint64_t v) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        a[i] = v;
}

__global__ void k_fill32(uint32_t *__restrict__ a, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) a[i] = 0;
}

__device__ __forceinline__ uint64_t hash_at(const uint4 *rs, uint64_t i) {
    const uint2 v = reinterpret_cast<const uint2 *>(rs)[2 * i];
    return (uint64_t)v.x | ((uint64_t)v.y << 32);
}

// Records a part may hold (48 KB of LDS), their mean at most (hashes are uniform:
// random parts stay within 5% of it, repeats need the room), and how many parts
// there may be (their counters are in LDS).
constexpr uint32_t PART_CAP = 3072, PART_MEAN = 2048, MAX_PART_BITS = 13;
constexpr uint32_t TILE_THREADS = 1024, TILE_EACH = 8, TILE_RECS = TILE_THREADS * TILE_EACH;

// The records (hash, sec) to their parts, by the top part_bits of the hash: part
// p's are parts[p PART_CAP ..] in any order, count[p] of them; those beyond
// PART_CAP are left out. A block counts its tile's parts in LDS, takes its places
// with one atomic a part, and writes.
__global__ __launch_bounds__(TILE_THREADS) void k_partition(const uint64_t *__restrict__ hash,
                                                            const uint64_t *__restrict__ sec, uint64_t n,
                                                            int part_bits, uint32_t *__restrict__ count,
                                                            uint4 *__restrict__ parts) {
    extern __shared__ uint32_t part_at[];
    const uint32_t np = 1u << part_bits;
    auto part_of = [&](uint64_t x) { return (uint32_t)(x >> 1 >> (63 - part_bits)); };
    for (uint32_t p = threadIdx.x; p < np; p += TILE_THREADS) part_at[p] = 0;
    __syncthreads();
    const uint64_t t0 = (uint64_t)blockIdx.x * TILE_RECS;
    uint64_t h[TILE_EACH];
    uint32_t rank[TILE_EACH];
#pragma unroll
    for (uint32_t u = 0; u < TILE_EACH; u++) {
        const uint64_t i = t0 + u * TILE_THREADS + threadIdx.x;
        h[u] = i < n ? hash[i] : 0;
    }
#pragma unroll
    for (uint32_t u = 0; u < TILE_EACH; u++)
        if (t0 + u * TILE_THREADS + threadIdx.x < n) rank[u] = atomicAdd(&part_at[part_of(h[u])], 1u);
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < np; p += TILE_THREADS) {
        const uint32_t c = part_at[p];
        if (c) part_at[p] = atomicAdd(&count[p], c);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < TILE_EACH; u++) {
        const uint64_t i = t0 + u * TILE_THREADS + threadIdx.x;
        if (i >= n) break;
        const uint32_t p = part_of(h[u]);
        const uint64_t s = sec[i];
        const uint64_t at = (uint64_t)part_at[p] + rank[u];
        if (at < PART_CAP)
            parts[(uint64_t)p * PART_CAP + at] =
                make_uint4((uint32_t)h[u], (uint32_t)(h[u] >> 32), (uint32_t)(s >> 32), (uint32_t)s);
    }
}

// order of (hash, position, packed)
__device__ __forceinline__ bool rec_less(const uint4 &a, const uint4 &b) {
    if (a.y != b.y) return a.y < b.y;
    if (a.x != b.x) return a.x < b.x;
    return a.z != b.z ? a.z < b.z : a.w < b.w;
}

// One part a block: its records to bins of LDS by the next hash bits (about one a
// bin), then each to its place in its bin by counting smaller records there.
constexpr uint32_t SORT_THREADS = 512, SORT_EACH = PART_CAP / SORT_THREADS, SORT_BIN_BITS = 11;
constexpr uint32_t SORT_BINS = 1u << SORT_BIN_BITS;

__global__ __launch_bounds__(SORT_THREADS) void k_sort_parts(const uint4 *__restrict__ parts,
                                                             const uint32_t *__restrict__ count,
                                                             const uint64_t *__restrict__ first, int part_bits,
                                                             uint4 *__restrict__ out, uint32_t *__restrict__ over) {
    __shared__ uint4 rec[PART_CAP];
    __shared__ uint32_t bins[SORT_BINS + 1];
    __shared__ uint32_t wave_tot[SORT_THREADS / 64];
    const uint32_t n = count[blockIdx.x], tid = threadIdx.x;
    if (n > PART_CAP) {
        if (tid == 0) *over = 1u;
        return;
    }
    const uint4 *in = parts + (uint64_t)blockIdx.x * PART_CAP;
    for (uint32_t t = tid; t <= SORT_BINS; t += SORT_THREADS) bins[t] = 0;
    __syncthreads();
    const int shift = 64 - part_bits - (int)SORT_BIN_BITS;
    auto bin_of = [&](const uint4 &r) {
        return (uint32_t)((((uint64_t)r.y << 32) | r.x) >> shift) & (SORT_BINS - 1);
    };
    uint4 r[SORT_EACH];
    uint32_t slot[SORT_EACH];
#pragma unroll
    for (uint32_t u = 0; u < SORT_EACH; u++)
        if (u * SORT_THREADS + tid < n) r[u] = in[u * SORT_THREADS + tid];
#pragma unroll
    for (uint32_t u = 0; u < SORT_EACH; u++)
        if (u * SORT_THREADS + tid < n) slot[u] = atomicAdd(&bins[bin_of(r[u])], 1u);
    __syncthreads();
    // counts to starts, four bins a thread
    constexpr uint32_t E = SORT_BINS / SORT_THREADS;
    uint32_t c[E], sum = 0;
#pragma unroll
    for (uint32_t u = 0; u < E; u++) sum += c[u] = bins[E * tid + u];
    const uint32_t incl = wave_incl_scan_dpp(sum);
    if (lane_id() == 63) wave_tot[tid / 64] = incl;
    __syncthreads();
    uint32_t at = incl - sum;
    for (uint32_t w = 0; w < tid / 64; w++) at += wave_tot[w];
#pragma unroll
    for (uint32_t u = 0; u < E; u++) {
        bins[E * tid + u] = at;
        at += c[u];
    }
    if (tid == SORT_THREADS - 1) bins[SORT_BINS] = at;
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < SORT_EACH; u++)
        if (u * SORT_THREADS + tid < n) rec[bins[bin_of(r[u])] + slot[u]] = r[u];
    __syncthreads();
    uint4 *dst = out + first[blockIdx.x];
    for (uint32_t i = tid; i < n; i += SORT_THREADS) {
        const uint4 x = rec[i];
        const uint32_t b = bin_of(x), b0 = bins[b], b1 = bins[b + 1];
        uint32_t place = b0;
        for (uint32_t j = b0; j < b1; j++) {
            const uint4 y = rec[j];
            place += rec_less(y, x) || (j < i && !rec_less(x, y)) ? 1u : 0u;
        }
        dst[place] = x;
    }
}

// A bucket start is written only where the hash changes: at change point i
// the buckets after the previous change point's bucket (all of them from 0
// when the previous run is the table's first) up to bucket(hash[i]) start at
// i, so the first hash's run is never inside a bucket (step2/index.cu:187-212).
__global__ void k_starts(const uint4 *__restrict__ rs, uint64_t n, int bits, uint64_t *__restrict__ starts) {
    const uint64_t h0 = n ? hash_at(rs, 0) : 0;
    for (uint64_t i = 1 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t h = hash_at(rs, i), hp = hash_at(rs, i - 1);
        if (h == hp) continue;
        const uint64_t top = h >> (64 - bits);
        const uint64_t lo = hp == h0 ? 0 : (hp >> (64 - bits)) + 1;
        for (uint64_t b = lo; b <= top; b++) starts[b] = i;
    }
}

// runs of equal hashes: hist[c] for c = 1..100, hist[101] for longer runs. Nearly
// every run is of one record: those are counted in registers, one LDS atomic a
// wave. Blocks add their bins to the same few words, ~13 ns apart whoever adds:
// 1024 blocks at most (8192 made this 107 us for 4.0 M records, now 31 us).
__global__ void k_runs(const uint4 *__restrict__ rs, uint64_t n, unsigned long long *__restrict__ hist) {
    __shared__ unsigned long long h[RUN_BINS];
    for (int t = threadIdx.x; t < RUN_BINS; t += blockDim.x) h[t] = 0;
    __syncthreads();
    uint32_t ones = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t v = hash_at(rs, i);
        if (i > 0 && hash_at(rs, i - 1) == v) continue;
        uint64_t j = i + 1;
        while (j < n && j - i <= 100 && hash_at(rs, j) == v) j++;
        const uint64_t c = j - i;
        if (c == 1) ones++;
        else atomicAdd(&h[c > 100 ? 101 : c], 1ull);
    }
    ones = wave_sum(ones);
    if (lane_id() == 0 && ones) atomicAdd(&h[1], (unsigned long long)ones);
    __syncthreads();
    for (int t = threadIdx.x; t < RUN_BINS; t += blockDim.x)
        if (h[t]) atomicAdd(&hist[t], h[t]);
}

unsigned grid_of(uint64_t n) {
    const uint64_t g = (n + 255) / 256;
    return (unsigned)(g < 8192 ? (g ? g : 1) : 8192);
}

void check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw BuildError{e, what};
}

}  // namespace

BuildArena::BuildArena(uint64_t estimate, void *&kept, uint64_t &kept_bytes)
    : next_(estimate), kept_(kept), kept_bytes_(kept_bytes) {
    if (kept_bytes_ >= estimate) {
        at_ = static_cast<char *>(kept_);
        left_ = kept_bytes_;
    } else if (kept_) {
        (void)hipFree(kept_);
        kept_ = nullptr;
        kept_bytes_ = 0;
    }
}

BuildArena::~BuildArena() {
    for (void *p : blocks_) (void)hipFree(p);
}

void *BuildArena::bytes(uint64_t n) {
    n = (std::max<uint64_t>(n, 1) + 255) & ~(uint64_t)255;
    if (n > left_) {
        uint64_t size = std::max(n, next_);
        void *p = nullptr;
        hipError_t e = hipMalloc(&p, size);
        if (e != hipSuccess && size > n) {  // no room for a large block: piece by piece
            (void)hipGetLastError();
            size = n;
            e = hipMalloc(&p, size);
        }
        check(e, "hipMalloc (index build)");
        if (!kept_ && size <= KEEP_MAX) {
            kept_ = p;
            kept_bytes_ = size;
        } else {
            blocks_.push_back(p);
        }
        at_ = static_cast<char *>(p);
        left_ = size;
        next_ = size > n ? size / 4 : 0;  // (the estimate fell short)
    }
    void *p = at_;
    at_ += n;
    left_ -= n;
    return p;
}

// the parts of n records
static int part_bits_of(uint64_t n) {
    int bits = 0;
    while ((n >> bits) > PART_MEAN) bits++;
    return bits;
}

uint64_t build_estimate(uint64_t bases, const gis_params &p) {
    const uint64_t recs = bases / (uint64_t)std::max(p.k - p.s + 1, 1) + bases / 64 + 65536;
    const int pb = part_bits_of(recs);
    // sequence, packed bases and N mask, window states twice; per syncmer
    // position and hash; per record the sort keys, and the parts or the sort's
    // other buffers and workspace
    return bases * 7 / 2 + recs * (16 + 16) +
           std::max<uint64_t>(recs * 16 + (16ull << 20) + bases / 8,
                              pb <= (int)MAX_PART_BITS ? ((uint64_t)PART_CAP * 16) << pb : 0);
}

// the two sorts of the library
static void sort_by_library(const RefSeeds &s, uint4 *rs, BuildArena &arena, hipStream_t st) {
    const uint64_t n = s.n;
    uint64_t *sec1 = arena.get<uint64_t>(n), *h1 = arena.get<uint64_t>(n);
    rocprim::double_buffer<uint64_t> sec(s.sec, sec1), hash(s.hash, h1);
    // stable by (position, packed), then stable by hash
    const unsigned lo = s.zeros ? 0u : 32u, hi = s.zeros ? 64u : 32u + (unsigned)s.pos_bits;
    size_t tb1 = 0, tb2 = 0;
    if (hi > lo)
        check(rocprim::radix_sort_pairs(nullptr, tb1, sec, hash, (size_t)n, lo, hi, st), "radix sort size");
    check(rocprim::radix_sort_pairs(nullptr, tb2, hash, sec, (size_t)n, 0, 64, st), "radix sort size");
    void *tmp = arena.bytes(std::max<size_t>(std::max(tb1, tb2), 1));
    if (hi > lo)
        check(rocprim::radix_sort_pairs(tmp, tb1, sec, hash, (size_t)n, lo, hi, st), "radix sort by position");
    check(rocprim::radix_sort_pairs(tmp, tb2, hash, sec, (size_t)n, 0, 64, st), "radix sort by hash");
    hipLaunchKernelGGL(k_pack, dim3(grid_of(n)), dim3(256), 0, st, rs, n, hash.current(), sec.current());
    check(hipGetLastError(), "index sort kernels");
}

void device_sort_records(const RefSeeds &s, uint4 *rs, BuildArena &arena, hipStream_t st) {
    const uint64_t n = s.n;
    if (n == 0) return;
    const int pb = part_bits_of(n);
    if (pb <= (int)MAX_PART_BITS) {
        const uint32_t np = 1u << pb;
        uint4 *parts = arena.get<uint4>((uint64_t)np * PART_CAP);
        uint32_t *count = arena.get<uint32_t>(np + 1);  // and the overflow word
        uint64_t *first = arena.get<uint64_t>(np + 1), *tmp = arena.get<uint64_t>(scan_tmp_words(np) + 8);
        hipLaunchKernelGGL(k_fill32, dim3(grid_of(np + 1)), dim3(256), 0, st, count, np + 1);
        hipLaunchKernelGGL(k_partition, dim3((unsigned)((n + TILE_RECS - 1) / TILE_RECS)), dim3(TILE_THREADS),
                           np * sizeof(uint32_t), st, s.hash, s.sec, n, pb, count, parts);
        launch_scan(count, first, np, tmp, st);
        hipLaunchKernelGGL(k_sort_parts, dim3(np), dim3(SORT_THREADS), 0, st, parts, count, first, pb, rs, count + np);
        check(hipGetLastError(), "index sort kernels");
        uint32_t over = 0;
        check(hipMemcpyAsync(&over, count + np, sizeof over, hipMemcpyDeviceToHost, st), "part overflow");
        check(hipStreamSynchronize(st), "index sort kernels");
        if (!over) return;
    }
    sort_by_library(s, rs, arena, st);
}

namespace {

// a table the lookups can trust: sorted by (hash, position), and every
// record inside [starts[b], starts[b + 1]) carries b in its top hash bits
__global__ void k_validate(const uint4 *__restrict__ rs, uint64_t n, const uint64_t *__restrict__ starts, int bits,
                           unsigned *__restrict__ bad) {
    const uint64_t nb = 1ull << bits;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n || i < nb;
         i += (uint64_t)gridDim.x * blockDim.x) {
        if (i >= 1 && i < n) {
            const uint4 a = rs[i - 1], c = rs[i];
            const uint64_t ha = (uint64_t)a.x | ((uint64_t)a.y << 32), hc = (uint64_t)c.x | ((uint64_t)c.y << 32);
            if (ha > hc || (ha == hc && a.z > c.z)) atomicOr(bad, 1u);
        }
        if (i < nb) {
            const uint64_t s = starts[i], e = starts[i + 1];
            if (s < e && e <= n &&
                ((hash_at(rs, s) >> (64 - bits)) != i || (hash_at(rs, e - 1) >> (64 - bits)) != i))
                atomicOr(bad, 2u);
        }
    }
}

}  // namespace

const char *device_validate_index(const uint4 *rs, uint64_t n, const uint64_t *starts, int bits, hipStream_t st) {
    unsigned *bad = nullptr;
    check(hipMalloc(&bad, sizeof(unsigned)), "hipMalloc");
    unsigned h = 0;
    hipError_t e = hipMemsetAsync(bad, 0, sizeof(unsigned), st);
    if (e == hipSuccess) {
        const uint64_t items = std::max<uint64_t>(n, 1ull << bits);
        hipLaunchKernelGGL(k_validate, dim3(grid_of(items)), dim3(256), 0, st, rs, n, starts, bits, bad);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&h, bad, sizeof(unsigned), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    (void)hipFree(bad);
    check(e, "index validation");
    if (h & 1u) return "randstrobes not sorted by (hash, position)";
    if (h & 2u) return "bucket starts do not match the records' hashes";
    return nullptr;
}

void device_finish_index(const uint4 *rs, uint64_t n, int bits, uint64_t *starts, uint64_t *hist_out,
                         BuildArena &arena, hipStream_t st) {
    const uint64_t nb = (1ull << bits) + 1;
    unsigned long long *hist = arena.get<unsigned long long>(RUN_BINS);
    hipLaunchKernelGGL(k_fill, dim3(grid_of(nb)), dim3(256), 0, st, starts, nb, n);
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(256), 0, st, reinterpret_cast<uint64_t *>(hist),
                       (uint64_t)RUN_BINS, (uint64_t)0);
    if (n > 1) hipLaunchKernelGGL(k_starts, dim3(grid_of(n)), dim3(256), 0, st, rs, n, bits, starts);
    if (n > 0) hipLaunchKernelGGL(k_runs, dim3(std::min(grid_of(n), 1024u)), dim3(256), 0, st, rs, n, hist);
    check(hipGetLastError(), "index starts and run histogram");
    check(hipMemcpyAsync(hist_out, hist, RUN_BINS * sizeof(uint64_t), hipMemcpyDeviceToHost, st), "run histogram");
    check(hipStreamSynchronize(st), "index starts and run histogram");
}

}  // namespace gis
