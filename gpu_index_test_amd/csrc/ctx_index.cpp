// C ABI: contexts and the resident strobemer index (StrobemerIndex,
// step2/index.hpp:37-183).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "driver_internal.h"
#include "host_copy.h"
#include "index_build.h"
#include "index_host.h"

using namespace gis;

namespace {

// the bucket lines of the resident table (one 128-byte line per bucket)
void build_lines(gis_ctx *ctx) {
    DevIndexStore &ix = ctx->ix;
    table_room<uint4>(ix.lines, (size_t)BUCKET_LINE << ix.bits);
    launch_bucket_lines(static_cast<const uint4 *>(ix.rs.p), static_cast<const uint64_t *>(ix.starts.p), ix.bits,
                        static_cast<uint4 *>(ix.lines.p), ctx->stream);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

// Loads a table in place of the resident one: load(keep) fills ix and returns false
// if it refuses the table. The memory of the table before, and of a build before,
// serves the load where it can, but must not be why one fails: a load that runs out
// of memory starts again with all of that given back, and keeps none (keep false).
// A load that fails for good leaves nothing behind.
template <typename F>
bool load_table(gis_ctx *ctx, F load) {
    DevIndexStore &ix = ctx->ix;
    drop_table(ix);
    for (bool keep = true;; keep = false) {
        HipError err{hipSuccess, ""};
        bool ok = false;
        struct Undo {
            gis_ctx *ctx;
            const bool &ok;
            ~Undo() {
                if (ok) return;
                (void)hipStreamSynchronize(ctx->stream);
                release_table(ctx->ix);
                release(ctx->build_mem);
            }
        };
        try {
            Undo undo{ctx, ok};
            if (!load(keep)) return false;
            build_lines(ctx);
            ok = true;
        } catch (const HipError &e) {
            err = e;
        } catch (const BuildError &e) {
            err = HipError{e.e, e.what};
        }
        if (ok) break;
        if (err.e != hipErrorOutOfMemory || !keep) throw err;
        (void)hipGetLastError();
    }
    ix.loaded = true;
    return true;
}

void upload_index(gis_ctx *ctx, const HostIndex &h) {
    DevIndexStore &ix = ctx->ix;
    load_table(ctx, [&](bool) {
        table_room<gis_ref_randstrobe>(ix.rs, h.rs.size());
        table_room<uint64_t>(ix.starts, h.starts.size());
        if (!h.rs.empty())
            HIP_CHECK(hipMemcpy(ix.rs.p, h.rs.data(), h.rs.size() * sizeof(gis_ref_randstrobe),
                                hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(ix.starts.p, h.starts.data(), h.starts.size() * 8, hipMemcpyHostToDevice));
        ix.n = h.rs.size();
        ix.bits = h.bits;
        ix.filter_cutoff = h.filter_cutoff;
        ix.params = h.params;
        ix.distinct = h.distinct_strobemers;
        ix.once = h.tot_occur_once;
        ix.high = h.tot_high_ab;
        ix.mid = h.tot_mid_ab;
        ix.index_cutoff = h.index_cutoff;
        return true;
    });
}

void download_index(gis_ctx *ctx, HostIndex &h) {
    const DevIndexStore &ix = ctx->ix;
    h.rs.resize(ix.n);
    h.starts.resize((1ULL << ix.bits) + 1);
    if (ix.n)
        HIP_CHECK(hipMemcpy(h.rs.data(), ix.rs.p, ix.n * sizeof(gis_ref_randstrobe), hipMemcpyDeviceToHost));
    HIP_CHECK(hipMemcpy(h.starts.data(), ix.starts.p, h.starts.size() * 8, hipMemcpyDeviceToHost));
    h.bits = ix.bits;
    h.filter_cutoff = ix.filter_cutoff;
    h.params = ix.params;
}

}  // namespace

extern "C" int gis_device_count(int *count) {
    if (!count) return GIS_ERR_BAD_PARAMETER;
    int c = 0;
    if (hipGetDeviceCount(&c) != hipSuccess) c = 0;
    *count = c;
    return GIS_OK;
}

extern "C" int gis_ctx_create(int device, gis_ctx **out) {
    if (!out) return GIS_ERR_BAD_PARAMETER;
    *out = nullptr;
    int c = 0;
    if (hipGetDeviceCount(&c) != hipSuccess || c <= 0) return GIS_ERR_HIP;
    if (device < 0 || device >= c) return GIS_ERR_BAD_PARAMETER;
    if (hipSetDevice(device) != hipSuccess) return GIS_ERR_HIP;
    // the allocation-free lookup's array address on this device; if it
    // cannot be had, that entry point reports it and the rest works on
    (void)noalloc_setup(device);
    gis_ctx *ctx = new gis_ctx();
    ctx->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess && prop.multiProcessorCount > 0)
        ctx->n_cu = prop.multiProcessorCount;
    // default-priority stream
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
        delete ctx;
        return GIS_ERR_HIP;
    }
    *out = ctx;
    return GIS_OK;
}

extern "C" void gis_ctx_destroy(gis_ctx *ctx) {
    if (!ctx) return;
    {
        std::lock_guard<std::recursive_mutex> lk(ctx->mu);
        (void)hipSetDevice(ctx->device);
        (void)hipStreamSynchronize(ctx->stream);
        batch_free(ctx->scratch);
        ctx->scratch = nullptr;
        for (gis_batch *b : ctx->lanes) batch_free(b);
        ctx->lanes.clear();
        dma_release(ctx->dma);
        ctx->dma = nullptr;
        pairwork_free(ctx->pairs);
        ctx->pairs = nullptr;
        release(ctx->ix.rs);
        release(ctx->ix.starts);
        release(ctx->ix.lines);
        release(ctx->build_mem);
        if (ctx->turn_ev) (void)hipEventDestroy(ctx->turn_ev);
        hostcopy_free(ctx->host_copy);
        ctx->host_copy = nullptr;
        (void)hipStreamDestroy(ctx->stream);
    }
    delete ctx;
}

extern "C" const char *gis_last_error(const gis_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

// contigs the 24-bit reference index and 32-bit positions of a record can hold
static int check_contigs(gis_ctx *ctx, const char *const *seqs, const uint64_t *lens, uint32_t n_refs) {
    if (n_refs && (!seqs || !lens)) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null argument");
    if (n_refs >= (1u << 24)) return fail(ctx, GIS_ERR_BAD_PARAMETER, "too many reference sequences for the 24-bit ref index");
    for (uint32_t j = 0; j < n_refs; j++) {
        if (lens[j] >= (1ull << 32)) return fail(ctx, GIS_ERR_BAD_PARAMETER, "reference sequence longer than 2^32 - 1");
        if (lens[j] && !seqs[j]) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null reference sequence");
    }
    return GIS_OK;
}

extern "C" int gis_index_build(gis_ctx *ctx, const char *const *seqs, const uint64_t *lens,
                               uint32_t n_refs, const gis_params *params, int bits, float f,
                               int n_threads) {
    (void)n_threads;  // the device seeds every contig
    API_BEGIN(ctx)
    if (!params) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null argument");
    if (int rc = check_contigs(ctx, seqs, lens, n_refs)) return rc;
    uint64_t total = 0;
    for (uint32_t j = 0; j < n_refs; j++) total += lens[j];
    if (total == 0) return fail(ctx, GIS_ERR_INVALID_FASTA, "No reference sequences found");
    if (bits == -1) bits = pick_bits(total, *params);
    if (bits < 8 || bits > 31) return fail(ctx, GIS_ERR_BAD_PARAMETER, "Bits must be between 8 and 31");
    DevIndexStore &ix = ctx->ix;
    load_table(ctx, [&](bool keep) {
        uint64_t hist[RUN_BINS] = {};
        uint64_t n = 0;
        DevBuf once;  // the build's memory if it is not to stay
        DevBuf &mem = keep ? ctx->build_mem : once;
        struct Release {
            DevBuf &b;
            ~Release() { release(b); }
        } release_once{once};
        {
            BuildArena arena(build_estimate(total, *params), mem.p, mem.bytes);
            const RefSeeds seeds = device_seed_reference(seqs, lens, n_refs, *params, true, arena, ctx->stream);
            n = seeds.n;
            uint4 *rs = table_room<uint4>(ix.rs, n);
            table_room<uint64_t>(ix.starts, (1ull << bits) + 1);
            device_sort_records(seeds, rs, arena, ctx->stream);
            device_finish_index(rs, n, bits, static_cast<uint64_t *>(ix.starts.p), hist, arena, ctx->stream);
        }
        HostIndex st;
        filter_stats(hist, f, st);
        ix.n = n;
        ix.bits = bits;
        ix.filter_cutoff = st.filter_cutoff;
        ix.params = *params;
        ix.distinct = st.distinct_strobemers;
        ix.once = st.tot_occur_once;
        ix.high = st.tot_high_ab;
        ix.mid = st.tot_mid_ab;
        ix.index_cutoff = st.index_cutoff;
        return true;
    });
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_reference_randstrobes(gis_ctx *ctx, const char *const *seqs, const uint64_t *lens,
                                         uint32_t n_refs, const gis_params *params, gis_ref_randstrobe *out,
                                         uint64_t capacity, uint64_t *n_out) {
    API_BEGIN(ctx)
    if (!params || !n_out) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null argument");
    if (int rc = check_contigs(ctx, seqs, lens, n_refs)) return rc;
    *n_out = 0;
    uint64_t total = 0;
    for (uint32_t j = 0; j < n_refs; j++) total += lens[j];
    if (total == 0) return GIS_OK;
    try {
        BuildArena arena(build_estimate(total, *params), ctx->build_mem.p, ctx->build_mem.bytes);
        const RefSeeds seeds = device_seed_reference(seqs, lens, n_refs, *params, false, arena, ctx->stream);
        const uint64_t n = seeds.n;
        *n_out = n;
        if (n > capacity || (n && !out))
            return fail(ctx, GIS_ERR_CAPACITY,
                        "record capacity " + std::to_string(capacity) + " < " + std::to_string(n));
        if (n) HIP_CHECK(hipMemcpy(out, seeds.recs, n * sizeof(gis_ref_randstrobe), hipMemcpyDeviceToHost));
    } catch (const BuildError &e) {
        throw HipError{e.e, e.what};
    }
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_index_upload(gis_ctx *ctx, const gis_ref_randstrobe *randstrobes, uint64_t n,
                                const uint64_t *starts, int bits, uint32_t filter_cutoff,
                                const gis_params *params) {
    API_BEGIN(ctx)
    if (!params || !starts || (n && !randstrobes)) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null argument");
    if (bits < 8 || bits > 31) return fail(ctx, GIS_ERR_BAD_PARAMETER, "Bits must be between 8 and 31");
    // the lookups and the hit order rely on the table's (hash, position) order
    for (uint64_t i = 1; i < n; i++) {
        const auto &a = randstrobes[i - 1], &c = randstrobes[i];
        if (a.hash > c.hash || (a.hash == c.hash && a.position > c.position))
            return fail(ctx, GIS_ERR_INVALID_INDEX, "randstrobes not sorted by (hash, position)");
    }
    const uint64_t nb = (1ULL << bits) + 1;
    for (uint64_t i = 0; i < nb; i++)
        if (starts[i] > n || (i && starts[i] < starts[i - 1]))
            return fail(ctx, GIS_ERR_INVALID_INDEX, "bucket starts out of range");
    HostIndex h;
    h.rs.assign(randstrobes, randstrobes + n);
    h.starts.assign(starts, starts + nb);
    h.bits = bits;
    h.filter_cutoff = filter_cutoff;
    h.params = *params;
    upload_index(ctx, h);
    return GIS_OK;
    API_END(ctx)
}

// .sti v2 (step2/index.cu:73-134) mapped into memory and copied from the
// mapping straight into HBM
extern "C" int gis_index_read_sti(gis_ctx *ctx, const char *path, const gis_params *expected) {
    API_BEGIN(ctx)
    if (!path) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null path");
    MappedSti m;
    std::string err;
    const int rc = map_sti(path, expected, m, err);
    if (rc) return fail(ctx, rc, err);
    const char *why = nullptr;
    try {
        DevIndexStore &ix = ctx->ix;
        load_table(ctx, [&](bool) {
            table_room<gis_ref_randstrobe>(ix.rs, m.n);
            table_room<uint64_t>(ix.starts, (1ull << m.bits) + 1);
            const uint64_t chunk = 256ull << 20;
            const char *src = reinterpret_cast<const char *>(m.rs);
            char *dst = static_cast<char *>(ix.rs.p);
            for (uint64_t o = 0, tot = m.n * sizeof(gis_ref_randstrobe); o < tot; o += chunk)
                HIP_CHECK(hipMemcpy(dst + o, src + o, std::min(chunk, tot - o), hipMemcpyHostToDevice));
            HIP_CHECK(hipMemcpy(ix.starts.p, m.starts, ((1ull << m.bits) + 1) * 8, hipMemcpyHostToDevice));
            // the file's table must be one the lookups can trust
            why = device_validate_index(static_cast<const uint4 *>(ix.rs.p), m.n,
                                        static_cast<const uint64_t *>(ix.starts.p), m.bits, ctx->stream);
            if (why) return false;
            ix.n = m.n;
            ix.bits = m.bits;
            ix.filter_cutoff = m.filter_cutoff;
            ix.params = m.params;
            ix.distinct = ix.once = ix.high = ix.mid = ix.index_cutoff = 0;
            return true;
        });
    } catch (...) {
        unmap_sti(m);
        throw;
    }
    unmap_sti(m);
    if (why) return fail(ctx, GIS_ERR_INVALID_INDEX, std::string("Index file has incorrect format: ") + why);
    return GIS_OK;
    API_END(ctx)
}

// .sti v2 written from HBM in chunks (no whole host copy of the table)
extern "C" int gis_index_write_sti(gis_ctx *ctx, const char *path) {
    API_BEGIN(ctx)
    if (!path) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null path");
    if (!ctx->ix.loaded) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    const DevIndexStore &ix = ctx->ix;
    FILE *fp = std::fopen(path, "wb");
    if (!fp) return fail(ctx, GIS_ERR_IO, std::string(path) + ": " + std::strerror(errno));
    bool ok = true;
    auto put = [&](const void *d, size_t n) { ok = ok && std::fwrite(d, 1, n, fp) == n; };
    put("STI\1", 4);
    const uint32_t version = 2;
    put(&version, 4);
    // a reserved chunk of 8 zero bytes, as the reference writes it
    const uint64_t reserved_size = 8, reserved = 0;
    put(&reserved_size, 8);
    put(&reserved, 8);
    const gis_params &p = ix.params;
    const int32_t v32[9] = {(int32_t)ix.filter_cutoff, ix.bits, p.canonical_read_length, p.k, p.s, p.l, p.u,
                            (int32_t)p.q, p.max_dist};
    put(v32, sizeof v32);
    put(&ix.n, 8);
    std::vector<char> buf;
    const uint64_t chunk = 256ull << 20;
    const uint64_t tot = ix.n * sizeof(gis_ref_randstrobe);
    try {
        buf.resize((size_t)std::min(chunk, std::max<uint64_t>(tot, 8)));
        for (uint64_t o = 0; o < tot && ok; o += chunk) {
            const uint64_t k = std::min(chunk, tot - o);
            HIP_CHECK(hipMemcpy(buf.data(), static_cast<const char *>(ix.rs.p) + o, k, hipMemcpyDeviceToHost));
            put(buf.data(), k);
        }
        const uint64_t nb = (1ull << ix.bits) + 1;
        put(&nb, 8);
        std::vector<uint64_t> st(nb);
        HIP_CHECK(hipMemcpy(st.data(), ix.starts.p, nb * 8, hipMemcpyDeviceToHost));
        put(st.data(), nb * 8);
    } catch (...) {
        std::fclose(fp);
        throw;
    }
    if (std::fclose(fp) != 0) ok = false;
    if (!ok) return fail(ctx, GIS_ERR_IO, std::string(path) + ": write failed");
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_index_info_get(gis_ctx *ctx, gis_index_info *out) {
    API_BEGIN(ctx)
    if (!out) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null output");
    if (!ctx->ix.loaded) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    const DevIndexStore &ix = ctx->ix;
    out->n_randstrobes = ix.n;
    out->bits = ix.bits;
    out->filter_cutoff = ix.filter_cutoff;
    out->params = ix.params;
    out->distinct_strobemers = ix.distinct;
    out->tot_occur_once = ix.once;
    out->tot_high_ab = ix.high;
    out->tot_mid_ab = ix.mid;
    out->index_cutoff = ix.index_cutoff;
    // (the table's; the arrays may be those of a larger one before it)
    out->device_bytes = std::max<uint64_t>(ix.n, 1) * sizeof(gis_ref_randstrobe) + ((1ull << ix.bits) + 1) * 8 +
                        ((uint64_t)BUCKET_LINE * sizeof(uint4) << ix.bits);
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_index_download(gis_ctx *ctx, gis_ref_randstrobe *randstrobes, uint64_t *starts) {
    API_BEGIN(ctx)
    if (!ctx->ix.loaded) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    const DevIndexStore &ix = ctx->ix;
    // (in stream order: a pinned array then takes them at the link's rate, 1.1 ms
    // for 64 MB, where hipMemcpy took 2.1 ms)
    if (randstrobes && ix.n)
        copy_to_host(ctx, randstrobes, ix.rs.p, ix.n * sizeof(gis_ref_randstrobe), ctx->stream);
    if (starts) copy_to_host(ctx, starts, ix.starts.p, ((1ULL << ix.bits) + 1) * 8, ctx->stream);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_fused_config_get(gis_ctx *ctx, gis_fused_config *out) {
    if (!ctx || !out) return GIS_ERR_BAD_PARAMETER;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    *out = ctx->fcfg;
    return GIS_OK;
}

extern "C" int gis_fused_config_set(gis_ctx *ctx, const gis_fused_config *cfg) {
    if (!ctx || !cfg) return GIS_ERR_BAD_PARAMETER;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    const gis_fused_config c = *cfg;
    if (c.waves_per_block != 2 && c.waves_per_block != 4 && c.waves_per_block != 8)
        return fail(ctx, GIS_ERR_BAD_PARAMETER, "waves_per_block must be 2, 4 or 8");
    if (c.length_split != 0 && c.length_split != 1)
        return fail(ctx, GIS_ERR_BAD_PARAMETER, "length_split must be 0 or 1");
    if (c.queue != 0 && c.queue != 1) return fail(ctx, GIS_ERR_BAD_PARAMETER, "queue must be 0 or 1");
    if (c.queue == 1 && (c.chunk < 1 || c.chunk > 4096))
        return fail(ctx, GIS_ERR_BAD_PARAMETER, "chunk must be in 1..4096");
    if (c.blocks_per_cu < 0 || c.blocks_per_cu > 64)
        return fail(ctx, GIS_ERR_BAD_PARAMETER, "blocks_per_cu must be in 0..64");
    if (c.queue == 1 && c.blocks_per_cu == 0)
        return fail(ctx, GIS_ERR_BAD_PARAMETER, "a dynamic queue needs a persistent grid (blocks_per_cu > 0)");
    ctx->fcfg = c;
    if (c.queue == 0) ctx->fcfg.chunk = 0;
    return GIS_OK;
}
