// Device half of strobemer index construction (StrobemerIndex::populate,
// step2/index.cu:143-244): sort the RefRandstrobe records by (hash,
// position, packed), fill the bucket starts with the reference's rule for
// where a bucket begins, and histogram the runs of equal hashes.
//
// The sort is two stable LSD radix sorts of the library (rocPRIM): first by
// position, then by hash. The records come in contig order, so equal (hash,
// position) stay in the order of their packed word without sorting by it, and a
// single contig's positions ascend already: 8 to 12 digit passes instead of 16
// (4.0 M records on 7 contigs: 538 us, before 740 us). The bucket starts and the histogram are plain
// grid-stride kernels over the sorted table.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>

#include "index_build.h"
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

__device__ __forceinline__ uint64_t hash_at(const uint4 *rs, uint64_t i) {
    const uint2 v = reinterpret_cast<const uint2 *>(rs)[2 * i];
    return (uint64_t)v.x | ((uint64_t)v.y << 32);
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
        blocks_.push_back(p);
        at_ = static_cast<char *>(p);
        left_ = size;
        next_ = size > n ? size / 4 : 0;  // (the estimate fell short)
    }
    void *p = at_;
    at_ += n;
    left_ -= n;
    return p;
}

uint64_t build_estimate(uint64_t bases, const gis_params &p) {
    const uint64_t recs = bases / (uint64_t)std::max(p.k - p.s + 1, 1) + bases / 64 + 65536;
    // sequence, packed bases and N mask, window states twice; per syncmer
    // position and hash; per record the sort's two double buffers; its workspace
    return bases * 7 / 2 + recs * (16 + 32) + (16ull << 20) + bases / 8;
}

void device_sort_records(const RefSeeds &s, uint4 *rs, BuildArena &arena, hipStream_t st) {
    const uint64_t n = s.n;
    if (n == 0) return;
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
