// Copies from HBM to a caller's arrays, in stream order. A pageable array of some
// size goes through pinned chunks of the context, emptied on the host while the next
// ones cross the link; the runtime's own way pins the array for each copy (20 MB of
// seeds: 1.44 ms, now 0.82; for arrays that the device reads it measured no worse
// than chunks, and stays). One transfer at a time has the chunks.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <vector>

#include "batch_internal.h"

namespace gis {

struct HostCopy;
void hostcopy_free(HostCopy *h);
// dst is complete when the stream is, or already on return (pageable)
void copy_to_host(gis_ctx *ctx, void *dst, const void *src, size_t n, hipStream_t st);

// Several arrays of some KB or MB to pinned arrays by one kernel, where a copy each
// takes ~15 us beside its bytes' time: true if all are pinned to their last byte and
// aligned for it, else nothing is done. (Offsets, fractions and flags of 65,536 reads beside their
// NAMs: 25 us, with a copy each 48.)
bool copy_small_to_host(const std::vector<CopyItem> &items, hipStream_t st);

// positions of keys, both pageable: the lookup reads its keys from the pinned chunks
// and writes their positions over them, across the link and while other chunks are
// filled and emptied on the host (10^6 keys: 790 us with a copy each way, now 440)
void lookup_through_host(gis_ctx *ctx, const uint64_t *keys, uint64_t n, uint64_t *positions, hipStream_t st);

// p points at memory that the runtime knows: its own copies take such arrays
bool pinned_array(const void *p);

// [p, p + bytes) lies in one pinned allocation (hipHostMalloc) that the GPU reaches
// at the same address: a copy engine or a kernel may read or write all of it
bool pinned_range(const void *p, size_t bytes);

}  // namespace gis
