// NAM consumer of paired reads: the reference order of each NAM list, pair
// classification, MAPQ and the joint NAM pairs (step2/main.cu:870-910,
// 1719-1830, 3449-3472, 3552-3581, 4641-4646).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/gis.h"

namespace gis {

// largest max_tries: the per-lane "NAM already paired" flags hold 256 bits
constexpr int PAIR_MAX_TRIES = 256;

// Device view of one pair step. Mate 1 of pair p is list p, mate 2 is list
// n_pairs + p of the 2 n_pairs NAM lists at off/in.
struct PairDev {
    const uint64_t *off;  // [2n+1]
    const gis_nam *in;    // input lists
    gis_nam *ord;         // lists in the reference order
    uint32_t n_pairs;
    int grouped;          // input lists sorted by (is_rc, ref_id): rank within a group range only
    uint8_t *types;       // [n]
    float *drop;          // [2n] top_dropoff
    uint8_t *mapq;        // [2n]
    uint32_t *tcnt;       // [5 * nblk] per block type counts, type-major
    const uint64_t *tpos; // [5 * nblk + 1] their exclusive scan
    uint32_t *tids;       // [n] pair ids grouped by type
    uint32_t nblk;
    gis_nam_pair *jtmp;   // entries at joint_place()
    const uint64_t *jplace; // [n+1] the pairs' places in jtmp (null: by a linear bound)
    // A pair of lists of c1 and c2 NAMs, M = 2 max_tries + 1, has at most
    // min(c1 c2, M) + c1 + c2 entries: at most c1 + c2 + jadd with jadd = M, and at
    // most c1 + c2 + (c1 + c2) jmul / 2^16 with jmul / 2^16 >= sqrt(M) / 2 (c1 c2 is at
    // most x^2, x = (c1 + c2) / 2, and min(x^2, M) at most x sqrt(M)). One of the two.
    uint64_t jmul, jadd;
    uint32_t *jcnt;       // [n]
    const uint64_t *joff; // [n+1]
    gis_nam_pair *jout;   // entries at joff
    uint64_t jout_cap;    // its room; a larger total leaves it as it is
    uint64_t *totals;     // [8], pinned host words: type starts in tids and their total, joint total, err
    unsigned *err;        // PAIR_ERR_* bits
    uint32_t *n_long;     // lists in longs; 0 between steps, like err
    uint32_t *longs;      // [2n] lists of more than 64 NAMs, in drop's memory before drop is written
    float dropoff, mu, sigma;
    int max_tries;
    int joint;
};

enum : unsigned { PAIR_ERR_DUPLICATE = 1, PAIR_ERR_JOINT = 2 };

constexpr unsigned PAIR_BLOCK = 256;

size_t pair_blocks(uint32_t n_pairs);
// reference order, types, dropoff, MAPQ and type lists
void launch_pairs_classify(const PairDev &P, uint64_t *scan_tmp, hipStream_t st);
// the pairs' places in jtmp by the exact bounds of their entries, their end in
// place[n]; jcnt is scratch for it
void launch_joint_bounds(const PairDev &P, uint64_t *place, uint64_t *scan_tmp, hipStream_t st);
// joint NAM pairs into jtmp, their counts scanned into joff, compacted into jout
void launch_pairs_joint(const PairDev &P, uint64_t *scan_tmp, hipStream_t st);
// the compaction again, with more room at jout
void launch_pairs_joint_compact(const PairDev &P, hipStream_t st);
// the step's totals and error bits to the host
void launch_pairs_totals(const PairDev &P, hipStream_t st);

}  // namespace gis
