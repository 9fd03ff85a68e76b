// Device half of strobemer index construction (index_build.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "../../include/gis.h"

namespace gis {

constexpr int RUN_BINS = 102;  // run-length histogram: [1..100] exact, [101] longer runs

struct BuildError {
    hipError_t e;
    const char *what;
};

// Device memory of one build: pieces cut from a few large blocks. An allocation
// and its release cost ~180 us together for a small block and ~600 us for the 400
// MB that 20 Mbp of reference take, so the first block is sized for the whole
// build, a second one is taken only where the estimate falls short, and the first
// one stays with the context (kept) for its next build if it is at most KEEP_MAX:
// a larger reference's build takes far longer than that. The others go with the
// arena.
class BuildArena {
  public:
    static constexpr uint64_t KEEP_MAX = 512ull << 20;
    BuildArena(uint64_t estimate, void *&kept, uint64_t &kept_bytes);
    ~BuildArena();
    BuildArena(const BuildArena &) = delete;
    BuildArena &operator=(const BuildArena &) = delete;
    void *bytes(uint64_t n);
    template <typename T>
    T *get(uint64_t n) {
        return static_cast<T *>(bytes(n * sizeof(T)));
    }

  private:
    std::vector<void *> blocks_;
    char *at_ = nullptr;
    uint64_t left_ = 0, next_;
    void *&kept_;
    uint64_t &kept_bytes_;
};

// device memory of a whole build of `bases` bases (a randstrobe in every k - s +
// 1 bases or so): sequence, windows, syncmers, records twice for the sort
uint64_t build_estimate(uint64_t bases, const gis_params &p);

// The RefRandstrobe records of every contig (RandstrobeGenerator over each
// contig, step2/randstrobes.cu:161-190, step2/index.cu:246-311), seeded on
// the device in (contig, position) order; contigs shorter than w_max get
// zero records in their slots. The arrays are the arena's.
struct RefSeeds {
    uint64_t n = 0;
    uint64_t *hash = nullptr;  // split form: hashes, and position << 32 | packed
    uint64_t *sec = nullptr;
    uint4 *recs = nullptr;     // else: records
    // sorting by the position bits alone (below 2^pos_bits) leaves records of
    // equal hash and position in the order of their packed word: they come in
    // contig order, one a contig and position. Zero records break that.
    int pos_bits = 0;
    bool zeros = false;
};
RefSeeds device_seed_reference(const char *const *seqs, const uint64_t *lens, uint32_t n_refs, const gis_params &p,
                               bool split, BuildArena &arena, hipStream_t st);
// the records of a split RefSeeds sorted by (hash, position, packed) into rs (n
// records); the seeds' arrays are used up
void device_sort_records(const RefSeeds &s, uint4 *rs, BuildArena &arena, hipStream_t st);
// checks a resident table and its starts: null if the lookups can trust
// them, else what is wrong (unsorted records, or bucket starts that do not
// match the records' top hash bits)
const char *device_validate_index(const uint4 *rs, uint64_t n, const uint64_t *starts, int bits, hipStream_t st);
// bucket starts (2^bits + 1 entries) and the run-length histogram of a
// sorted table; hist_out receives RUN_BINS host counters
void device_finish_index(const uint4 *rs, uint64_t n, int bits, uint64_t *starts, uint64_t *hist_out,
                         BuildArena &arena, hipStream_t st);

}  // namespace gis
