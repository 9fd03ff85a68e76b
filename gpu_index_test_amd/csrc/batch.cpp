// C ABI: device batches and the whole-path / stage entry points.
//
// A batch holds reads resident in HBM and every buffer of the path. A run is
// a fixed sequence of launches on the context's stream with no host round
// trip: variable-size intermediates (hits, rescue hits) are placed by device
// scans of per-read counts and checked against their capacity on the device,
// and the single synchronisation at the end reads the totals and the
// overflow bits. When an array was too small it grows to the total the scan
// reported and the batch runs again; results never depend on it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <mutex>
#include <vector>

#include "batch_internal.h"
#include "host_copy.h"

using namespace gis;

namespace gis {

gis_batch *batch_new(gis_ctx *ctx, Workspace *share) {
    gis_batch *b = new gis_batch();
    b->ctx = ctx;
    b->stream = ctx->stream;
    b->ws = share ? share : new Workspace();
    b->ws->refs++;
    return b;
}

gis_batch *batch_new_stream(gis_ctx *ctx) {
    gis_batch *b = batch_new(ctx, nullptr);
    // default priority, like the context's stream; the workspace owns it, so
    // batches sharing the workspace keep it while any of them lives
    if (hipStreamCreateWithFlags(&b->ws->stream, hipStreamNonBlocking) != hipSuccess) {
        b->ws->stream = nullptr;
        batch_free(b);
        throw HipError{hipErrorOutOfMemory, "hipStreamCreateWithFlags"};
    }
    b->stream = b->ws->stream;
    return b;
}

// the device arrays of a workspace, and of a batch's own inputs
static std::vector<DevBuf *> ws_bufs(Workspace *w) {
    return {&w->long_scratch, &w->rs_cnt, &w->rs_nfwd, &w->rs_hash, &w->rs_span,
            &w->sy_cnt, &w->sy_hash, &w->sy_pos, &w->pos, &w->hcnt, &w->rcnt, &w->lk_bytes, &w->lk_stream,
            &w->hit_total, &w->rhit_total, &w->frac, &w->flags, &w->nam_cnt, &w->hit_off,
            &w->rhit_off, &w->hits, &w->rhits, &w->keys, &w->rkeys, &w->nam_ws, &w->rnam_ws,
            &w->nam_fin, &w->rnam_fin, &w->nam_slots, &w->nam_off, &w->nams_out, &w->scan_tmp,
            &w->ctl, &w->spill_ids, &w->gwork, &w->split_list, &w->sel_ids, &w->seeds};
}

static std::vector<DevBuf *> input_bufs(gis_batch *b) {
    return {&b->seqs, &b->read_off, &b->read_len, &b->rs_off, &b->sy_off, &b->long_off, &b->queue};
}

static void workspace_release(Workspace *w) {
    for (DevBuf *x : ws_bufs(w)) release(*x);
    if (w->h_ctl) (void)hipHostFree(w->h_ctl);
    pairwork_free(w->pairs);
    if (w->stream) (void)hipStreamDestroy(w->stream);
    delete w;
}

uint64_t batch_device_bytes(gis_batch *b) {
    uint64_t t = 0;
    for (DevBuf *x : input_bufs(b)) t += x->bytes;
    for (DevBuf *x : ws_bufs(b->ws)) t += x->bytes;
    return t;
}

static void graph_drop(gis_batch::GraphEntry &g) {
    for (int part = 0; part < 3; part++) {
        if (g.exec[part]) (void)hipGraphExecDestroy(g.exec[part]);
        if (g.graph[part]) (void)hipGraphDestroy(g.graph[part]);
        g.exec[part] = nullptr;
        g.graph[part] = nullptr;
    }
}

void batch_trim(gis_batch *b) {
    HIP_CHECK(hipStreamSynchronize(b->stream));
    for (auto &g : b->graphs) graph_drop(g);
    b->graphs.clear();
    for (DevBuf *x : input_bufs(b)) release(*x);
    for (DevBuf *x : ws_bufs(b->ws)) release(*x);
    b->ws->hit_cap = b->ws->rhit_cap = b->ws->out_cap = 0;
    b->ws->merge_scratch = false;
    b->ws->owner = nullptr;
    b->ran = false;
    b->n_reads = 0;
}

void batch_free(gis_batch *b) {
    if (!b) return;
    for (DevBuf *x : input_bufs(b)) release(*x);
    for (auto &e : b->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto &g : b->graphs) graph_drop(g);
    if (b->ws) {
        if (b->ws->owner == b) b->ws->owner = nullptr;
        if (b->ws->in_flight == b) {
            b->ws->in_flight = nullptr;
            b->ctx->launched--;
        }
        if (--b->ws->refs == 0) workspace_release(b->ws);
    }
    delete b;
}

}  // namespace gis

namespace gis {

// reads up to this length form the fused kernel's short bin
constexpr int SHORT_BIN = 160;

// long-read scratch bytes of the seeding stage for one read of length L
// (layout of long_bufs in kernels.hip)
uint64_t long_bytes(uint64_t L) {
    auto a8 = [](uint64_t x) { return (x + 7) & ~7ULL; };
    return 16 * L + 8 * (L / 64 + 2) + a8(4 * L) + a8(L) + a8(L) + 64;
}

// Small host calls (at most SMALL_READS reads and SMALL_BYTES of input): inputs
// go through h_in and one kernel, results through h_out, so a call is its
// launches and one wait. Larger calls gain more from the copy engines.
constexpr uint32_t SMALL_READS = 4096;
constexpr size_t SMALL_BYTES = 1u << 20;

static size_t a16(size_t x) { return (x + 15) & ~(size_t)15; }

// NAMs up to which the results of a small call go through h_out (4 MB of them): with
// more, the copy engines are the faster way
constexpr uint64_t HOST_NAMS_MAX = (4u << 20) / sizeof(gis_nam);

// the places of a small call's results in h_out
struct HostOut {
    uint64_t *off;
    float *frac;
    uint8_t *flags;
    gis_nam *nams;
    uint64_t nam_cap;
    size_t bytes;
};

static HostOut host_out(gis_batch *b) {
    const size_t n = b->n_reads;
    HostOut h;
    const size_t o_frac = a16(8 * (n + 1)), o_flags = o_frac + a16(4 * n), o_nams = o_flags + a16(n);
    h.nam_cap = std::max<uint64_t>(16 * n + 1024, b->ws->host_nams);
    h.bytes = o_nams + sizeof(gis_nam) * h.nam_cap;
    uint8_t *p = b->ws->h_out.data();
    h.off = reinterpret_cast<uint64_t *>(p);
    h.frac = reinterpret_cast<float *>(p + o_frac);
    h.flags = p + o_flags;
    h.nams = reinterpret_cast<gis_nam *>(p + o_nams);
    return h;
}

// Whether a small call's results go to h_out: not where the calls before had too many
// NAMs a read for it. (A call that finds out by itself runs twice.)
static bool host_out_wanted(gis_batch *b) {
    if (b->n_reads == 0 || (uint64_t)b->nams_a_read * b->n_reads > HOST_NAMS_MAX) return false;
    b->ws->h_out.resize(host_out(b).bytes);
    return true;
}

// more NAMs than h_out had room for, tot in all: it keeps that room from now on, or
// they go the large way. True if h_out holds them now.
static bool host_out_grow(gis_batch *b, uint64_t tot) {
    const uint64_t need = tot + tot / 8;
    b->host_out = need <= HOST_NAMS_MAX;
    if (!b->host_out) return false;
    b->ws->host_nams = std::max(b->ws->host_nams, need);
    b->ws->h_out.resize(host_out(b).bytes);
    return true;
}

// the NAMs of a finished run, for the calls after it
static void note_nams(gis_batch *b) {
    const uint64_t n = b->n_reads, tot = b->ws->tot_nams;
    if (n) b->nams_a_read = std::max<uint64_t>((tot + n - 1) / n, b->nams_a_read / 2);
}

// all of `items` through h_in and one launch on the batch's stream (and the
// control block cleared, with ctl); the batch's earlier work has been waited for
static void copy_in_small(gis_batch *b, const std::vector<CopyItem> &items, DevCtl *ctl) {
    CopyList c{};
    size_t at = 0;
    for (const CopyItem &i : items) at += a16(i.bytes);
    b->h_in.resize(at + 16);
    at = 0;
    for (const CopyItem &i : items) {
        if (!i.bytes) continue;
        std::memcpy(b->h_in.data() + at, i.src, i.bytes);
        c.src[c.n] = b->h_in.data() + at;
        c.dst[c.n] = i.dst;
        c.bytes[c.n] = (uint32_t)i.bytes;
        c.block[c.n + 1] = c.block[c.n] + (uint32_t)((i.bytes + CopyList::BLOCK_BYTES - 1) / CopyList::BLOCK_BYTES);
        c.n++;
        at += a16(i.bytes);
    }
    launch_copy_in(c, ctl, b->stream);
}

// Enqueue staged inputs; true when they went the small way. The caller's arrays
// are read until the stream has been waited for.
static bool copy_in(gis_batch *b, const std::vector<CopyItem> &items) {
    size_t bytes = 0;
    for (const CopyItem &i : items) bytes += i.bytes;
    const bool small = b->n_reads <= SMALL_READS && bytes <= SMALL_BYTES && items.size() <= CopyList::MAX;
    if (small) copy_in_small(b, items, nullptr);
    else
        for (const CopyItem &c : items)
            HIP_CHECK(hipMemcpyAsync(c.dst, c.src, c.bytes, hipMemcpyHostToDevice, b->stream));
    return small;
}

DevBatch make_devbatch(gis_batch *b) {
    DevBatch d{};
    d.seqs = static_cast<const char *>(b->seqs.p);
    d.read_off = static_cast<const uint64_t *>(b->read_off.p);
    d.read_len = static_cast<const uint32_t *>(b->read_len.p);
    d.n_reads = b->n_reads;
    d.rs_off = static_cast<const uint64_t *>(b->rs_off.p);
    d.rs_cnt = static_cast<uint32_t *>(b->ws->rs_cnt.p);
    d.rs_nfwd = static_cast<uint32_t *>(b->ws->rs_nfwd.p);
    d.rs_hash = static_cast<uint64_t *>(b->ws->rs_hash.p);
    d.rs_span = static_cast<uint32_t *>(b->ws->rs_span.p);
    d.sy_off = static_cast<const uint64_t *>(b->sy_off.p);
    d.sy_cnt = static_cast<uint32_t *>(b->ws->sy_cnt.p);
    d.sy_hash = static_cast<uint64_t *>(b->ws->sy_hash.p);
    d.sy_pos = static_cast<uint64_t *>(b->ws->sy_pos.p);
    d.pos = static_cast<uint64_t *>(b->ws->pos.p);
    d.hcnt = static_cast<uint32_t *>(b->ws->hcnt.p);
    d.rcnt = static_cast<uint32_t *>(b->ws->rcnt.p);
    d.lk_bytes = static_cast<uint32_t *>(b->ws->lk_bytes.p);
    d.lk_stream = static_cast<uint32_t *>(b->ws->lk_stream.p);
    d.hit_total = static_cast<uint32_t *>(b->ws->hit_total.p);
    d.rhit_total = static_cast<uint32_t *>(b->ws->rhit_total.p);
    d.frac = static_cast<float *>(b->ws->frac.p);
    d.flags = static_cast<uint8_t *>(b->ws->flags.p);
    d.nam_cnt = static_cast<uint32_t *>(b->ws->nam_cnt.p);
    d.hit_off = static_cast<uint64_t *>(b->ws->hit_off.p);
    d.rhit_off = static_cast<uint64_t *>(b->ws->rhit_off.p);
    d.hits = static_cast<DevHit *>(b->ws->hits.p);
    d.rhits = static_cast<DevHit *>(b->ws->rhits.p);
    d.hit_cap = b->ws->hit_cap;
    d.rhit_cap = b->ws->rhit_cap;
    d.keys = static_cast<uint64_t *>(b->ws->keys.p);
    d.rkeys = static_cast<uint64_t *>(b->ws->rkeys.p);
    d.nam_ws = static_cast<WideNam *>(b->ws->nam_ws.p);
    d.rnam_ws = static_cast<WideNam *>(b->ws->rnam_ws.p);
    d.merge_scratch = b->ws->merge_scratch ? 1u : 0u;
    d.gwork = static_cast<uint4 *>(b->ws->gwork.p);
    d.gwork_cap = (uint32_t)std::min<uint64_t>(b->ws->gwork.bytes / sizeof(uint4), UINT32_MAX);
    d.split_list = static_cast<uint4 *>(b->ws->split_list.p);
    d.sel_ids = static_cast<uint32_t *>(b->ws->sel_ids.p);
    d.nam_fin = static_cast<gis_nam *>(b->ws->nam_fin.p);
    d.rnam_fin = static_cast<gis_nam *>(b->ws->rnam_fin.p);
    d.nam_slots = static_cast<gis_nam *>(b->ws->nam_slots.p);
    d.nam_off = static_cast<uint64_t *>(b->ws->nam_off.p);
    d.nams_out = static_cast<gis_nam *>(b->ws->nams_out.p);
    d.out_cap = b->ws->out_cap;
    d.long_off = static_cast<const uint64_t *>(b->long_off.p);
    d.long_scratch = static_cast<uint8_t *>(b->ws->long_scratch.p);
    d.ctl = static_cast<DevCtl *>(b->ws->ctl.p);
    d.spill_ids = static_cast<uint32_t *>(b->ws->spill_ids.p);
    if (b->host_out) {
        const HostOut h = host_out(b);
        d.nams_out = h.nams;
        d.out_cap = h.nam_cap;
        d.h_off = h.off;
        d.h_frac = h.frac;
        d.h_flags = h.flags;
    }
    return d;
}

// the batch's own per-read input arrays
void ensure_input_arrays(gis_batch *b, uint32_t n) {
    ensure<uint64_t>(b->read_off, n);
    ensure<uint32_t>(b->read_len, n);
    ensure<uint64_t>(b->rs_off, n + 1);
    ensure<uint64_t>(b->sy_off, n + 1);
    ensure<uint64_t>(b->long_off, n + 1);
    ensure<uint32_t>(b->queue, n);
}

// per-read arrays of the workspace
void ensure_read_arrays(gis_batch *b, uint32_t n) {
    ensure<uint32_t>(b->ws->rs_cnt, n);
    ensure<uint32_t>(b->ws->rs_nfwd, n);
    ensure<uint32_t>(b->ws->sy_cnt, n);
    ensure<uint32_t>(b->ws->lk_bytes, n);
    ensure<uint32_t>(b->ws->lk_stream, n);
    ensure<uint32_t>(b->ws->hit_total, n);
    ensure<uint32_t>(b->ws->rhit_total, n);
    ensure<uint32_t>(b->ws->nam_cnt, n);
    ensure<float>(b->ws->frac, n);
    ensure<uint8_t>(b->ws->flags, n);
    ensure<uint64_t>(b->ws->hit_off, n + 1);
    ensure<uint64_t>(b->ws->rhit_off, n + 1);
    ensure<uint64_t>(b->ws->nam_off, n + 1);
    ensure<uint64_t>(b->ws->scan_tmp, scan_tmp_words(n) + 8);
    ensure<DevCtl>(b->ws->ctl, 1);
    ensure<uint32_t>(b->ws->spill_ids, n);
    ensure<uint4>(b->ws->split_list, n);
    ensure<uint32_t>(b->ws->sel_ids, 3ull * n + 3);
    if (!b->ws->h_ctl) {
        HIP_CHECK(hipHostMalloc((void **)&b->ws->h_ctl, sizeof(DevCtl)));
        HIP_CHECK(hipHostGetDevicePointer((void **)&b->ws->h_ctl_dev, b->ws->h_ctl, 0));
    }
}

void ensure_slot_arrays(gis_batch *b, uint64_t slots) {
    ensure<uint64_t>(b->ws->rs_hash, slots);
    ensure<uint32_t>(b->ws->rs_span, slots);
    ensure<uint64_t>(b->ws->pos, slots);
    ensure<uint32_t>(b->ws->hcnt, slots);
    ensure<uint32_t>(b->ws->rcnt, slots);
}

// hit arrays, merge scratch and the NAM output (capacities in hits / NAMs)
void ensure_pools(gis_batch *b, uint64_t hit_cap, uint64_t rhit_cap, uint64_t out_cap) {
    b->ws->hit_cap = std::max(b->ws->hit_cap, hit_cap);
    b->ws->rhit_cap = std::max(b->ws->rhit_cap, rhit_cap);
    b->ws->out_cap = std::max(b->ws->out_cap, out_cap);
    ensure<DevHit>(b->ws->hits, b->ws->hit_cap);
    ensure<gis_nam>(b->ws->nam_fin, b->ws->hit_cap);
    ensure<DevHit>(b->ws->rhits, b->ws->rhit_cap);
    ensure<gis_nam>(b->ws->rnam_fin, b->ws->rhit_cap);
    if (b->ws->merge_scratch) {
        // merge scratch of reads beyond the merge's LDS budget, allocated
        // once a run has met such a read
        ensure<uint64_t>(b->ws->keys, 2 * b->ws->hit_cap);
        ensure<WideNam>(b->ws->nam_ws, b->ws->hit_cap);
        ensure<uint64_t>(b->ws->rkeys, 2 * b->ws->rhit_cap);
        ensure<WideNam>(b->ws->rnam_ws, b->ws->rhit_cap);
        // a split read of h > 64 hits has at most h / ITEM_HITS + 1 work items,
        // fewer than h / 48
        ensure<uint4>(b->ws->gwork, (b->ws->hit_cap + b->ws->rhit_cap) / 48 + 64);
    }
    ensure<gis_nam>(b->ws->nams_out, b->ws->out_cap);
}

void mark(gis_batch *b, const char *name) {
    if (b->n_ev >= 16) return;
    if (!b->ev[b->n_ev]) HIP_CHECK(hipEventCreate(&b->ev[b->n_ev]));
    HIP_CHECK(hipEventRecord(b->ev[b->n_ev], b->stream));
    b->ev_names.push_back(name);
    b->n_ev++;
}

// Stage reads into the batch: randstrobe-slot capacities and offsets come
// from the lengths, computed here once.
int batch_stage(gis_batch *b, const char *seqs, const uint64_t *offsets, const uint32_t *lens,
                uint32_t n, bool want_sy, uint64_t base, hipEvent_t before, std::vector<CopyItem> *defer,
                bool want_queue) {
    gis_ctx *ctx = b->ctx;
    if (!ctx->ix.loaded && !b->seed_params) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    if (n > 0 && (!seqs || !offsets || !lens)) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null read arrays");
    const gis_params &p = b->seed_params ? *b->seed_params : ctx->ix.params;
    uint64_t span = 0;
    b->h_rs_off.resize(n + 1);
    b->h_sy_off.resize(n + 1);
    b->h_long_off.resize(n + 1);
    b->h_read_off.resize(n);
    b->h_rs_off[0] = b->h_sy_off[0] = b->h_long_off[0] = 0;
    b->any_long = false;
    uint64_t rs_at = 0, sy_at = 0, long_at = 0;
    uint32_t n_long = 0;
    for (uint32_t r = 0; r < n; r++) {
        const uint64_t L = lens[r];
        if (L > GIS_MAX_READ_LEN)
            return fail(ctx, GIS_ERR_BAD_PARAMETER,
                        "read " + std::to_string(r) + " longer than " + std::to_string(GIS_MAX_READ_LEN));
        if (offsets[r] < base) return fail(ctx, GIS_ERR_BAD_PARAMETER, "read offset below the staged base");
        const uint64_t o = offsets[r] - base;
        b->h_read_off[r] = o;
        span = std::max(span, o + L);
        const int64_t nk = (int64_t)L - p.k + 1;
        const int64_t nf = nk - (int64_t)p.w_min;
        const uint64_t cap_sy = nk > 0 ? (uint64_t)nk : 0;
        const uint64_t cap_rs = (nf > 0 && L >= p.w_max) ? 2 * (uint64_t)nf : 0;
        rs_at += cap_rs;
        sy_at += cap_sy;
        const bool lg = L > (uint64_t)LMAX_LDS;
        b->any_long |= lg;
        long_at += lg ? long_bytes(L) : 0;
        n_long += L > (uint64_t)SHORT_BIN ? 1u : 0u;
        b->h_rs_off[r + 1] = rs_at;
        b->h_sy_off[r + 1] = sy_at;
        b->h_long_off[r + 1] = long_at;
    }
    b->n_reads = n;
    b->staged++;
    b->host_out = false;
    b->want_sy = want_sy;
    b->n_long = n_long;
    b->queue_ok = want_queue;
    // the fused kernel's work queue: read ids by length, longest first
    // (counting sort over lengths capped at 1023; stable within a length)
    if (want_queue) {
        uint32_t cnt[1025] = {};
        for (uint32_t r = 0; r < n; r++) cnt[1023 - std::min<uint32_t>(lens[r], 1023u) + 1]++;
        for (int i = 1; i < 1025; i++) cnt[i] += cnt[i - 1];
        b->h_queue.resize(n);
        for (uint32_t r = 0; r < n; r++) b->h_queue[cnt[1023 - std::min<uint32_t>(lens[r], 1023u)]++] = r;
    }
    ensure_input_arrays(b, n);
    b->tot_rs_cap = b->h_rs_off[n];
    b->span = span;
    ensure<char>(b->seqs, span + SEQ_PAD);
    std::vector<CopyItem> items;
    std::vector<CopyItem> &in = defer ? *defer : items;
    if (span) in.push_back({b->seqs.p, seqs + base, span});
    if (n) {
        in.push_back({b->read_off.p, b->h_read_off.data(), 8ull * n});
        in.push_back({b->read_len.p, lens, 4ull * n});
    }
    in.push_back({b->rs_off.p, b->h_rs_off.data(), 8ull * (n + 1)});
    // (read by the seeding for these alone)
    if (want_sy) in.push_back({b->sy_off.p, b->h_sy_off.data(), 8ull * (n + 1)});
    if (b->any_long) in.push_back({b->long_off.p, b->h_long_off.data(), 8ull * (n + 1)});
    if (n && want_queue) in.push_back({b->queue.p, b->h_queue.data(), 4ull * n});
    b->ran = false;
    if (defer) return GIS_OK;
    hipStream_t st = b->stream;
    if (before) HIP_CHECK(hipEventRecord(before, st));
    for (const CopyItem &c : items) HIP_CHECK(hipMemcpyAsync(c.dst, c.src, c.bytes, hipMemcpyHostToDevice, st));
    return GIS_OK;
}

int batch_upload(gis_batch *b, const char *seqs, const uint64_t *offsets, const uint32_t *lens,
                 uint32_t n, bool want_sy) {
    const int rc = batch_stage(b, seqs, offsets, lens, n, want_sy, 0, nullptr);
    if (rc) return rc;
    HIP_CHECK(hipStreamSynchronize(b->stream));
    return GIS_OK;
}

uint32_t rescue_cutoff_of(const gis_ctx *ctx, const gis_map_options &o) {
    // step2/main.cu:4204: R < 100 ? R * filter_cutoff : 100
    return o.rescue_level < 100 ? (uint32_t)(o.rescue_level * (int)ctx->ix.filter_cutoff) : 100u;
}

// The launch sequence of one run, enqueued on the context's stream.
// Stage events are recorded only for runs without graphs.
void enqueue_run(gis_batch *b, const RunOpts &r) {
    const int mode = r.mode, rescue_mode = r.rescue_mode, stop = r.stop;
    const uint32_t rcut = r.rcut, hard = r.hard;
    const auto mark = [&](gis_batch *x, const char *name) {
        if (!r.graph) gis::mark(x, name);
    };
    gis_ctx *ctx = b->ctx;
    hipStream_t st = b->stream;
    const DevIndex ix = dev_index(ctx);
    const SeedParams sp = make_seed_params(b->seed_params ? *b->seed_params : ctx->ix.params);
    const DevBatch d = make_devbatch(b);
    const uint32_t n = b->n_reads;
    uint64_t *tmp = static_cast<uint64_t *>(b->ws->scan_tmp.p);
    const bool front = r.part != PART_BACK, back = r.part != PART_FRONT;
    if (front) {
        b->n_ev = 0;
        b->ev_names.clear();
        mark(b, "start");
    }
    ReadSet set{nullptr, nullptr, n};
    const bool fused = mode == GIS_MODE_FUSED && stop == STOP_NONE;
    if (fused && front) {
        launch_reset_ctl(d.ctl, st);
        const gis_fused_config &fc = ctx->fcfg;
        const unsigned grid = fc.blocks_per_cu > 0 ? (unsigned)(ctx->n_cu * fc.blocks_per_cu) : 0u;
        const uint32_t chunk = fc.queue ? (uint32_t)fc.chunk : 0u;
        const uint32_t *q = static_cast<const uint32_t *>(b->queue.p);
        bool ok;
        if (fc.length_split) {
            ok = launch_fused(d, ix, sp, rcut, hard, q, b->n_long, 320, fc.waves_per_block, grid, chunk,
                              &d.ctl->q_head[0], st) &&
                 launch_fused(d, ix, sp, rcut, hard, q + b->n_long, n - b->n_long, SHORT_BIN,
                              fc.waves_per_block, grid, chunk, &d.ctl->q_head[1], st);
        } else {
            ok = launch_fused(d, ix, sp, rcut, hard, q, n, 320, fc.waves_per_block, grid, chunk,
                              &d.ctl->q_head[0], st);
        }
        if (!ok) throw HipError{hipErrorInvalidValue, "unsupported fused configuration"};
        mark(b, "fused");
    }
    if (fused) set = ReadSet{d.spill_ids, &d.ctl->n_spill, n};
    if (fused ? back : front) {
        launch_seed(d, set, sp, b->want_sy ? 1 : 0, b->any_long ? 1 : 0, fused ? 0 : 1, st);
        mark(b, "seed");
        launch_lookup(d, set, ix, rescue_mode, st);
        mark(b, "lookup");
    }
    if (!back) return;
    launch_hits(d, ix, rcut, hard, st);
    mark(b, "hits");
    if (stop == STOP_NONE) {
        launch_merge(d, set, st);
        mark(b, "merge");
        launch_output(d, fused ? 1 : 0, tmp, b->ws->h_ctl_dev, st);
        mark(b, "output");
    } else {
        launch_ctl_to_host(d, b->ws->h_ctl_dev, st);
    }
}

// size the workspace for this batch's reads (grow-only; cheap when it
// already fits)
void prepare_workspace(gis_batch *b) {
    const uint32_t n = b->n_reads;
    ensure_read_arrays(b, n);
    ensure_slot_arrays(b, b->tot_rs_cap);
    if (b->want_sy) {
        ensure<uint64_t>(b->ws->sy_hash, b->h_sy_off[n]);
        ensure<uint64_t>(b->ws->sy_pos, b->h_sy_off[n]);
    }
    if (b->any_long) ensure<uint8_t>(b->ws->long_scratch, b->h_long_off[n]);
    // initial pools: about the hits of typical reads (~0.16 per base), grown
    // on demand to what a run's scans report.
    // GIS_TEST_SMALL_POOLS starts them tiny so tests exercise the overflow path.
    // the hit array holds a HIT_REGION-hit region per read, then the pool of
    // the reads with more hits
    const uint64_t regions = (uint64_t)HIT_REGION * n;
    if (const char *e = std::getenv("GIS_TEST_SMALL_POOLS"); e && *e == '1')
        ensure_pools(b, regions + 64, 64, 16);
    else
        ensure_pools(b, regions + 4ull * n + b->span / 64 + 4096, 4ull * n + 4096, 12ull * n + 1024);
}

RunOpts run_opts(const gis_batch *b, const gis_map_options &o, int rescue_mode, int stop) {
    RunOpts r;
    r.mode = o.mode;
    r.rescue_mode = rescue_mode;
    r.rcut = rescue_cutoff_of(b->ctx, o);
    r.hard = o.hard_cutoff;
    r.stop = stop;
    r.graph = stop == STOP_NONE && (o.flags & GIS_RUN_NO_GRAPH) == 0;
    return r;
}

// Configurations whose graphs a batch keeps. Reads of uneven length make one of each
// batch that a stream's lane maps (the reads beyond SHORT_BIN are counted), and files
// mapped in turn come back to them: 400,000 such reads in batches of 32,768 on four
// lanes, fused, took 4710 us with 8 kept and 4410 with 16.
constexpr size_t GRAPHS_KEPT = 16;

// the launches of r (or of its part), by its captured graph where it has one
static void launch_part(gis_batch *b, const RunOpts &r) {
    gis_ctx *ctx = b->ctx;
    hipStream_t st = b->stream;
    if (r.graph) {
        bool replay = true;
        const DevBatch key = make_devbatch(b);
        // (launch arguments beside it; a seeding call may have moved the scan's alone)
        const void *const args[2] = {b->ws->scan_tmp.p, b->queue.p};
        const gis_fused_config &fc = ctx->fcfg;
        const int cfg[11] = {r.mode, r.rescue_mode, (int)r.rcut, (int)r.hard, r.stop,
                             (b->want_sy ? 1 : 0) | (b->any_long ? 2 : 0), fc.waves_per_block,
                             fc.length_split, fc.chunk, fc.blocks_per_cu, (int)b->n_long};
        gis_batch::GraphEntry *hit = nullptr;
        for (auto &g : b->graphs)
            if (std::memcmp(&key, &g.key, sizeof key) == 0 && std::memcmp(args, g.args, sizeof args) == 0 &&
                std::memcmp(cfg, g.cfg, sizeof cfg) == 0)
                hit = &g;
        if (!hit) {
            if (b->graphs.size() >= GRAPHS_KEPT) {
                auto old = b->graphs.begin();
                for (auto it = b->graphs.begin(); it != b->graphs.end(); ++it)
                    if (it->used < old->used) old = it;
                HIP_CHECK(hipStreamSynchronize(st));
                graph_drop(*old);
                b->graphs.erase(old);
            }
            gis_batch::GraphEntry e{};
            e.key = key;
            std::memcpy(e.args, args, sizeof args);
            e.epoch = ctx->ix.epoch;
            std::memcpy(e.cfg, cfg, sizeof cfg);
            b->graphs.push_back(e);
            hit = &b->graphs.back();
            replay = !b->lazy_graph;
        }
        hit->used = ++b->graph_clock;
        if (replay && !hit->exec[r.part]) {
            hipGraph_t g = nullptr;
            HIP_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            try {
                enqueue_run(b, r);
            } catch (...) {
                (void)hipStreamEndCapture(st, &g);
                if (g) (void)hipGraphDestroy(g);
                throw;
            }
            HIP_CHECK(hipStreamEndCapture(st, &g));
            const hipError_t ie = hipGraphInstantiate(&hit->exec[r.part], g, nullptr, nullptr, 0);
            if (ie != hipSuccess) {
                (void)hipGraphDestroy(g);
                hit->exec[r.part] = nullptr;
                throw HipError{ie, "hipGraphInstantiate"};
            }
            hit->graph[r.part] = g;
        }
        if (replay) HIP_CHECK(hipGraphLaunch(hit->exec[r.part], st));
        else enqueue_run(b, r);
    } else {
        enqueue_run(b, r);
    }
    HIP_CHECK(hipGetLastError());
}

// Enqueue one run on the batch's stream. With r.graph the launch sequence is
// captured once per configuration (buffers, mode, cutoffs, fused launch
// configuration) and replayed, a run in two parts by graphs of its own; a batch
// keeps the graphs of its last GRAPHS_KEPT configurations.
//
// in_turn (a burst: runs launched on streams of their own onto an idle device, none
// waited for yet): a large plain batch starts after the front of the one before it,
// its seeding and lookup (fused kernels are nearly the whole run: two batches of
// 60,000 took 1463 us in turn and 1370 to 1382 without). Launched together they would
// share the device from their first kernel and end together, and the first one's
// copies back could not run beside the others' kernels. (Three batches of 65,536
// reads of 150 bp and their results: 1797 us, side by side 2046.) Later launches
// find the runs out of step already, and side by side their phases fill the device
// better: 4 lanes without copies took 321 M reads/s against 291 M with turns kept
// throughout. A batch of fewer than TURN_READS does not fill the device and runs
// beside the others as it did.
constexpr uint32_t TURN_READS = 16384;
void batch_launch(gis_batch *b, const RunOpts &r, bool in_turn) {
    gis_ctx *ctx = b->ctx;
    hipStream_t st = b->stream;
    // (first: arrays of the workspace may move, also where a later one finds no memory)
    b->ws->owner = b;
    b->ran = false;
    b->last_run = RunId{b->staged, ctx->ix.epoch, r.rcut, r.hard};
    prepare_workspace(b);
    if (r.mode == GIS_MODE_FUSED && r.stop == STOP_NONE) {
        if (!b->queue_ok) throw HipError{hipErrorInvalidValue, "fused run of reads staged without the work queue"};
        ensure<gis_nam>(b->ws->nam_slots, (size_t)b->n_reads * F_NAMCAP);
    }
    // graphs captured against a table that has since been dropped hold its
    // freed addresses and old parameters: never replay them
    bool stale = false;
    for (const auto &g : b->graphs) stale |= g.epoch != ctx->ix.epoch;
    if (stale) {
        HIP_CHECK(hipStreamSynchronize(st));
        for (auto it = b->graphs.begin(); it != b->graphs.end();) {
            if (it->epoch == ctx->ix.epoch) {
                ++it;
                continue;
            }
            graph_drop(*it);
            it = b->graphs.erase(it);
        }
    }
    if (!in_turn || b->n_reads < TURN_READS || st == ctx->stream || r.mode == GIS_MODE_FUSED) {
        launch_part(b, r);
        return;
    }
    if (!ctx->turn_ev) HIP_CHECK(hipEventCreateWithFlags(&ctx->turn_ev, hipEventDisableTiming));
    if (ctx->turn_st && ctx->turn_st != st) HIP_CHECK(hipStreamWaitEvent(st, ctx->turn_ev, 0));
    RunOpts p = r;
    p.part = PART_FRONT;
    launch_part(b, p);
    HIP_CHECK(hipEventRecord(ctx->turn_ev, st));
    ctx->turn_st = st;
    p.part = PART_BACK;
    launch_part(b, p);
}

bool batch_ready(const gis_batch *b) { return hipStreamQuery(b->stream) == hipSuccess; }

// wait for the run on the stream; returns the overflow bits
static unsigned finish_once(gis_batch *b, const RunOpts &r) {
    HIP_CHECK(hipStreamSynchronize(b->stream));
    const bool fused = r.mode == GIS_MODE_FUSED && r.stop == STOP_NONE;
    b->ws->n_spill = fused ? b->ws->h_ctl->n_spill : 0;
    b->ws->tot_nams = r.stop == STOP_NONE ? b->ws->h_ctl->tot[2] : 0;
    return b->ws->h_ctl->overflow;
}

void batch_complete(gis_batch *b, const RunOpts &r) {
    unsigned ovf = finish_once(b, r);
    for (int attempt = 1; ovf && attempt < 6; attempt++) {
        // after a hit overflow the merges did not run, and after a merge
        // without its scratch some reads are missing, so the NAM total is
        // not final: grow what overflowed now and size the output next time
        if (ovf & (OVF_HITS | OVF_RHITS | OVF_MERGE)) ovf &= ~(unsigned)OVF_OUT;
        if (ovf & OVF_MERGE) b->ws->merge_scratch = true;
        if ((ovf & OVF_OUT) && b->host_out && host_out_grow(b, b->ws->tot_nams)) ovf &= ~(unsigned)OVF_OUT;
        ensure_pools(b, (ovf & OVF_HITS) ? b->ws->h_ctl->tot[0] + b->ws->h_ctl->tot[0] / 8 + 4096 : 0,
                     (ovf & OVF_RHITS) ? b->ws->h_ctl->tot[1] + b->ws->h_ctl->tot[1] / 8 + 4096 : 0,
                     (ovf & OVF_OUT) ? b->ws->tot_nams + b->ws->tot_nams / 8 + 1024 : 0);
        batch_launch(b, r);
        ovf = finish_once(b, r);
    }
    if (ovf) throw HipError{hipErrorOutOfMemory, "batch arrays still too small after regrowth"};
    b->last_mode = r.mode;
    b->last_graph = r.graph;
    b->ran = r.stop == STOP_NONE;
    if (!b->ran) return;
    b->last_run.over = true;
    note_nams(b);
}

void batch_run(gis_batch *b, const gis_map_options &o, int rescue_mode, int stop) {
    const RunOpts r = run_opts(b, o, rescue_mode, stop);
    batch_launch(b, r);
    batch_complete(b, r);
}

int batch_download(gis_batch *b, gis_nam_out *out) {
    gis_ctx *ctx = b->ctx;
    if (!out) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null output");
    if (!b->ran) return fail(ctx, GIS_ERR_STATE, "batch has not been run");
    if (b->ws->owner != b)
        return fail(ctx, GIS_ERR_STATE, "another batch sharing the workspace ran since this batch's run");
    const uint32_t n = b->n_reads;
    out->n_nams = b->ws->tot_nams;
    if (out->nam_capacity < b->ws->tot_nams || (b->ws->tot_nams && !out->nams))
        return fail(ctx, GIS_ERR_CAPACITY,
                    "NAM capacity " + std::to_string(out->nam_capacity) + " < " + std::to_string(b->ws->tot_nams));
    hipStream_t st = b->stream;
    if (b->host_out) {
        const HostOut h = host_out(b);
        if (out->nam_offsets) std::memcpy(out->nam_offsets, h.off, 8ull * (n + 1));
        if (b->ws->tot_nams) std::memcpy(out->nams, h.nams, sizeof(gis_nam) * b->ws->tot_nams);
        if (out->nonrepetitive_fraction && n) std::memcpy(out->nonrepetitive_fraction, h.frac, 4ull * n);
        if (out->flags && n) std::memcpy(out->flags, h.flags, n);
        return GIS_OK;
    }
    std::vector<CopyItem> small;
    if (out->nam_offsets) small.push_back({out->nam_offsets, b->ws->nam_off.p, 8ull * (n + 1)});
    if (out->nonrepetitive_fraction && n) small.push_back({out->nonrepetitive_fraction, b->ws->frac.p, 4ull * n});
    if (out->flags && n) small.push_back({out->flags, b->ws->flags.p, n});
    if (!copy_small_to_host(small, st))
        for (const CopyItem &c : small) copy_to_host(ctx, c.dst, c.src, c.bytes, st);
    if (b->ws->tot_nams) copy_to_host(ctx, out->nams, b->ws->nams_out.p, sizeof(gis_nam) * b->ws->tot_nams, st);
    HIP_CHECK(hipStreamSynchronize(st));
    return GIS_OK;
}

gis_batch *scratch_batch(gis_ctx *ctx) {
    if (!ctx->scratch) {
        ctx->scratch = batch_new(ctx, nullptr);
        ctx->scratch->lazy_graph = true;
    }
    return ctx->scratch;
}

gis_map_options opts_or_default(const gis_map_options *opt) {
    gis_map_options o;
    if (opt) o = *opt;
    else gis_map_options_default(&o);
    if (o.mode != GIS_MODE_FUSED) o.mode = GIS_MODE_PLAIN;
    return o;
}

}  // namespace gis

// ---------------- stage entry points ----------------

static_assert(sizeof(gis_query_randstrobe) == 24 && sizeof(gis_syncmer) == 16, "the records the device writes");

// Seeds of every read (query randstrobes, or syncmers) into out, dense and in
// read order; seeding parameters of the batch's seed_params or the index. The
// caller holds the context's lock.
static int seeds_of(gis_ctx *ctx, const gis_params *params, bool syncmers, const char *seqs, const uint64_t *offsets,
                    const uint32_t *lens, uint32_t n, uint64_t *out_offsets, void *out, uint64_t capacity,
                    uint64_t *n_out) {
    gis_batch *b = scratch_batch(ctx);
    struct Reset {
        gis_batch *b;
        ~Reset() { b->seed_params = nullptr; }
    } reset{b};
    b->seed_params = params;
    std::vector<CopyItem> items;
    if (int rc = batch_stage(b, seqs, offsets, lens, n, syncmers, 0, nullptr, &items, false)) return rc;
    Workspace *w = b->ws;
    ensure_read_arrays(b, n);
    ensure_slot_arrays(b, b->tot_rs_cap);
    if (syncmers) {
        ensure<uint64_t>(w->sy_hash, b->h_sy_off[n]);
        ensure<uint64_t>(w->sy_pos, b->h_sy_off[n]);
    }
    if (b->any_long) ensure<uint8_t>(w->long_scratch, b->h_long_off[n]);
    w->owner = b;
    b->ran = false;
    hipStream_t st = b->stream;
    StreamGuard guard{st};
    const bool small = copy_in(b, items);
    const DevBatch d = make_devbatch(b);
    uint64_t *off = d.nam_off, *tmp = static_cast<uint64_t *>(w->scan_tmp.p);
    launch_seed(d, ReadSet{nullptr, nullptr, n}, make_seed_params(params ? *params : ctx->ix.params), syncmers ? 1 : 0,
                b->any_long ? 1 : 0, 0, st);
    launch_scan(syncmers ? d.sy_cnt : d.rs_cnt, off, n, tmp, st);
    HIP_CHECK(hipGetLastError());
    const size_t rec = syncmers ? sizeof(gis_syncmer) : sizeof(gis_query_randstrobe);
    const uint64_t most = syncmers ? b->h_sy_off[n] : b->tot_rs_cap;
    // a small call's records go straight to pinned memory, as many as its slots
    // hold at most; a large one's are counted first
    const bool direct = small && n > 0 && most * rec <= 2 * SMALL_BYTES;
    uint64_t total = 0;
    if (direct) {
        const size_t head = a16(8ull * (n + 1));
        w->h_out.resize(head + most * rec);
        uint64_t *h_off = reinterpret_cast<uint64_t *>(w->h_out.data());
        launch_emit_seeds(d, syncmers ? 1 : 0, off, w->h_out.data() + head, h_off, st);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipStreamSynchronize(st));
        guard.armed = false;
        total = h_off[n];
    } else {
        HIP_CHECK(hipMemcpyAsync(&w->h_ctl->tot[2], off + n, 8, hipMemcpyDeviceToHost, st));
        HIP_CHECK(hipStreamSynchronize(st));
        total = w->h_ctl->tot[2];
    }
    if (n_out) *n_out = total;
    if (total > capacity || (total && !out))
        return fail(ctx, GIS_ERR_CAPACITY, syncmers ? "syncmer capacity too small" : "randstrobe capacity too small");
    if (direct) {
        if (total) std::memcpy(out, w->h_out.data() + a16(8ull * (n + 1)), total * rec);
        if (out_offsets) std::memcpy(out_offsets, w->h_out.data(), 8ull * (n + 1));
        return GIS_OK;
    }
    if (total) {
        ensure<char>(w->seeds, total * rec);
        launch_emit_seeds(d, syncmers ? 1 : 0, off, w->seeds.p, nullptr, st);
        HIP_CHECK(hipGetLastError());
        copy_to_host(ctx, out, w->seeds.p, total * rec, st);
    }
    if (out_offsets) copy_to_host(ctx, out_offsets, off, 8ull * (n + 1), st);
    HIP_CHECK(hipStreamSynchronize(st));
    return GIS_OK;
}

extern "C" int gis_syncmers_batch(gis_ctx *ctx, const char *seqs, const uint64_t *offsets,
                                  const uint32_t *lens, uint32_t n_reads, uint64_t *out_offsets,
                                  gis_syncmer *out, uint64_t capacity, uint64_t *n_out) {
    API_BEGIN(ctx)
    return seeds_of(ctx, nullptr, true, seqs, offsets, lens, n_reads, out_offsets, out, capacity, n_out);
    API_END(ctx)
}

extern "C" int gis_randstrobes_batch(gis_ctx *ctx, const char *seqs, const uint64_t *offsets,
                                     const uint32_t *lens, uint32_t n_reads, uint64_t *out_offsets,
                                     gis_query_randstrobe *out, uint64_t capacity, uint64_t *n_out) {
    API_BEGIN(ctx)
    return seeds_of(ctx, nullptr, false, seqs, offsets, lens, n_reads, out_offsets, out, capacity, n_out);
    API_END(ctx)
}

extern "C" int gis_randstrobes_params(gis_ctx *ctx, const gis_params *params, const char *seqs,
                                      const uint64_t *offsets, const uint32_t *lens, uint32_t n_reads,
                                      uint64_t *out_offsets, gis_query_randstrobe *out, uint64_t capacity,
                                      uint64_t *n_out) {
    API_BEGIN(ctx)
    if (!params) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null parameters");
    gis_params chk;
    if (gis_params_make(params->canonical_read_length, params->k, params->s, params->l, params->u,
                        (int)params->q, params->max_dist, &chk) != GIS_OK ||
        chk.t_syncmer != params->t_syncmer || chk.w_min != params->w_min || chk.w_max != params->w_max)
        return fail(ctx, GIS_ERR_BAD_PARAMETER, "invalid index parameters");
    return seeds_of(ctx, params, false, seqs, offsets, lens, n_reads, out_offsets, out, capacity, n_out);
    API_END(ctx)
}

extern "C" int gis_lookup_batch(gis_ctx *ctx, const uint64_t *hashes, uint64_t n, uint64_t *positions) {
    API_BEGIN(ctx)
    if (!ctx->ix.loaded) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    if (n && (!hashes || !positions)) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null argument");
    if (n == 0) return GIS_OK;
    // (overlapping arrays: all keys are read before a position is written)
    const bool apart = positions + n <= hashes || hashes + n <= positions;
    if (apart && !pinned_array(hashes) && !pinned_array(positions)) {
        lookup_through_host(ctx, hashes, n, positions, ctx->stream);
        return GIS_OK;
    }
    gis_batch *b = scratch_batch(ctx);
    uint64_t *dh = ensure<uint64_t>(b->ws->rs_hash, n);
    uint64_t *dp = ensure<uint64_t>(b->ws->pos, n);
    HIP_CHECK(hipMemcpyAsync(dh, hashes, 8 * n, hipMemcpyHostToDevice, ctx->stream));
    launch_find_flat(dev_index(ctx), dh, n, dp, ctx->stream);
    HIP_CHECK(hipGetLastError());
    copy_to_host(ctx, positions, dp, 8 * n, ctx->stream);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return GIS_OK;
    API_END(ctx)
}

static int copy_hits_out(gis_ctx *ctx, gis_batch *b, uint64_t *out_offsets, gis_hit *out,
                         uint64_t capacity, uint64_t *n_out) {
    const uint32_t n = b->n_reads;
    std::vector<uint8_t> flags(n);
    std::vector<uint64_t> ho(n), rho(n);
    std::vector<uint32_t> hcount(n), rcount(n);
    if (n) {
        HIP_CHECK(hipMemcpy(flags.data(), b->ws->flags.p, n, hipMemcpyDeviceToHost));
        HIP_CHECK(hipMemcpy(hcount.data(), b->ws->hit_total.p, 4ull * n, hipMemcpyDeviceToHost));
        HIP_CHECK(hipMemcpy(rcount.data(), b->ws->rhit_total.p, 4ull * n, hipMemcpyDeviceToHost));
        HIP_CHECK(hipMemcpy(ho.data(), b->ws->hit_off.p, 8ull * n, hipMemcpyDeviceToHost));
        HIP_CHECK(hipMemcpy(rho.data(), b->ws->rhit_off.p, 8ull * n, hipMemcpyDeviceToHost));
    }
    const uint64_t nh = n ? b->ws->h_ctl->tot[0] : 0, nrh = n ? b->ws->h_ctl->tot[1] : 0;
    std::vector<DevHit> h(nh), rh(nrh);
    if (nh) HIP_CHECK(hipMemcpy(h.data(), b->ws->hits.p, sizeof(DevHit) * nh, hipMemcpyDeviceToHost));
    if (nrh) HIP_CHECK(hipMemcpy(rh.data(), b->ws->rhits.p, sizeof(DevHit) * nrh, hipMemcpyDeviceToHost));
    uint64_t total = 0;
    // a read's hits: its region or pool place (hit_off) and count (hit_total);
    // rescued reads: their place in the rescue array
    for (uint32_t r = 0; r < n; r++) total += (flags[r] & GIS_FLAG_RESCUED) ? rcount[r] : hcount[r];
    if (n_out) *n_out = total;
    if (total > capacity || (total && !out)) return fail(ctx, GIS_ERR_CAPACITY, "hit capacity too small");
    uint64_t o = 0;
    std::vector<uint64_t> idx;
    for (uint32_t r = 0; r < n; r++) {
        if (out_offsets) out_offsets[r] = o;
        const bool resc = (flags[r] & GIS_FLAG_RESCUED) != 0;
        const std::vector<DevHit> &src = resc ? rh : h;
        const uint64_t lo = resc ? rho[r] : ho[r], hi = lo + (resc ? rcount[r] : hcount[r]);
        // group by (strand, ref) keeping the emission order inside a group
        idx.clear();
        for (uint64_t i = lo; i < hi; i++) idx.push_back(((uint64_t)src[i].ref_strand << 32) | (i - lo));
        std::sort(idx.begin(), idx.end());
        for (uint64_t key : idx) {
            const DevHit &x = src[lo + (uint32_t)key];
            gis_hit g;
            g.query_start = x.query_start;
            g.query_end = x.query_end;
            g.ref_start = x.ref_start;
            g.ref_end = x.ref_end;
            g.ref_id = (int32_t)(x.ref_strand & 0x7fffffffu);
            g.is_rc = (int32_t)(x.ref_strand >> 31);
            out[o++] = g;
        }
    }
    if (out_offsets) out_offsets[n] = o;
    return GIS_OK;
}

extern "C" int gis_hits_batch(gis_ctx *ctx, const char *seqs, const uint64_t *offsets,
                              const uint32_t *lens, uint32_t n_reads, const gis_map_options *opt,
                              uint64_t *out_offsets, gis_hit *out, uint64_t capacity, uint64_t *n_out) {
    API_BEGIN(ctx)
    gis_map_options o = opts_or_default(opt);
    o.mode = GIS_MODE_PLAIN;
    gis_batch *b = scratch_batch(ctx);
    int rc = batch_upload(b, seqs, offsets, lens, n_reads, false);
    if (rc) return rc;
    batch_run(b, o, 0, STOP_HITS);
    return copy_hits_out(ctx, b, out_offsets, out, capacity, n_out);
    API_END(ctx)
}

extern "C" int gis_find_nams_batch(gis_ctx *ctx, const char *seqs, const uint64_t *offsets,
                                   const uint32_t *lens, uint32_t n_reads, const gis_map_options *opt,
                                   gis_nam_out *out) {
    API_BEGIN(ctx)
    const gis_map_options o = opts_or_default(opt);
    gis_batch *b = scratch_batch(ctx);
    std::vector<CopyItem> items;
    const int rc = batch_stage(b, seqs, offsets, lens, n_reads, false, 0, nullptr, &items, o.mode == GIS_MODE_FUSED);
    if (rc) return rc;
    StreamGuard guard{b->stream};
    b->host_out = copy_in(b, items) && host_out_wanted(b);
    batch_run(b, o, 0, STOP_NONE);
    guard.armed = false;
    return batch_download(b, out);
    API_END(ctx)
}

// find_nams / find_nams_rescue over given query randstrobes on the context's
// scratch batch (the caller holds the context's lock)
static int qrs_run(gis_ctx *ctx, const gis_query_randstrobe *qrs, const uint64_t *query_offsets,
                   uint32_t n_queries, int rescue, uint32_t rescue_cutoff, uint32_t hard_cutoff, gis_nam_out *out) {
    if (!ctx->ix.loaded) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    if (!query_offsets || !out) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null argument");
    gis_batch *b = scratch_batch(ctx);
    const uint32_t n = n_queries;
    // each read's queries laid out forward strand first, each strand by (start, end, hash)
    const uint64_t total = query_offsets[n];
    // the arrays that the seeding would have left, built in pinned memory
    const size_t o_sp = a16(8 * total), o_cnt = o_sp + a16(4 * total), o_nf = o_cnt + a16(4ull * n),
                 o_off = o_nf + a16(4ull * n), in_bytes = o_off + 8ull * (n + 1);
    b->h_in.resize(in_bytes + 16);
    uint8_t *in = b->h_in.data();
    uint64_t *hh = reinterpret_cast<uint64_t *>(in), *off = reinterpret_cast<uint64_t *>(in + o_off);
    uint32_t *sp = reinterpret_cast<uint32_t *>(in + o_sp), *cnt = reinterpret_cast<uint32_t *>(in + o_cnt),
             *nf = reinterpret_cast<uint32_t *>(in + o_nf);
    std::vector<uint64_t> ord;
    for (uint32_t r = 0; r < n; r++) {
        const uint64_t lo = query_offsets[r], hi = query_offsets[r + 1];
        ord.clear();
        for (uint64_t i = lo; i < hi; i++) ord.push_back(i);
        std::stable_sort(ord.begin(), ord.end(), [&](uint64_t a, uint64_t c) {
            const auto &x = qrs[a], &y = qrs[c];
            if (x.is_reverse != y.is_reverse) return x.is_reverse < y.is_reverse;
            if (x.start != y.start) return x.start < y.start;
            if (x.end != y.end) return x.end < y.end;
            return x.hash < y.hash;
        });
        uint32_t f = 0;
        for (uint64_t j = 0; j < ord.size(); j++) {
            const auto &q = qrs[ord[j]];
            if (q.end > GIS_MAX_READ_LEN) return fail(ctx, GIS_ERR_BAD_PARAMETER, "query end too large");
            hh[lo + j] = q.hash;
            sp[lo + j] = span_pack((uint32_t)q.start, (uint32_t)q.end);
            if (!q.is_reverse) f++;
        }
        cnt[r] = (uint32_t)(hi - lo);
        nf[r] = f;
        off[r] = lo;
    }
    off[n] = total;
    b->n_reads = n;
    b->want_sy = false;
    b->any_long = false;
    // the per-read randstrobe offsets are the one input array the stages
    // after seeding read (a fresh context's scratch batch has none yet)
    ensure<uint64_t>(b->rs_off, (size_t)n + 1);
    ensure_read_arrays(b, n);
    ensure_slot_arrays(b, total);
    b->ws->owner = b;
    b->ran = false;
    ensure_pools(b, (uint64_t)HIT_REGION * n + 16ull * n + 4096, 16ull * n + 4096, 16ull * n + 1024);
    b->tot_rs_cap = total;
    const bool small = n > 0 && n <= SMALL_READS && in_bytes <= SMALL_BYTES;
    b->host_out = small && host_out_wanted(b);
    hipStream_t st = ctx->stream;
    StreamGuard guard{st};
    const CopyItem items[] = {{b->ws->rs_hash.p, hh, 8 * total},
                              {b->ws->rs_span.p, sp, 4 * total},
                              {b->ws->rs_cnt.p, cnt, 4ull * n},
                              {b->ws->rs_nfwd.p, nf, 4ull * n},
                              {b->rs_off.p, off, 8ull * (n + 1)}};
    if (small) {
        CopyList c{};
        for (const CopyItem &i : items) {
            if (!i.bytes) continue;
            c.src[c.n] = i.src;
            c.dst[c.n] = i.dst;
            c.bytes[c.n] = (uint32_t)i.bytes;
            c.block[c.n + 1] = c.block[c.n] + (uint32_t)((i.bytes + CopyList::BLOCK_BYTES - 1) / CopyList::BLOCK_BYTES);
            c.n++;
        }
        launch_copy_in(c, static_cast<DevCtl *>(b->ws->ctl.p), st);
    } else {
        for (const CopyItem &i : items)
            if (i.bytes) HIP_CHECK(hipMemcpyAsync(i.dst, i.src, i.bytes, hipMemcpyHostToDevice, st));
    }
    // the stages after seeding, with the rescue decision forced either way
    const DevIndex ix = dev_index(ctx);
    const ReadSet set{nullptr, nullptr, n};
    uint64_t *tmp = static_cast<uint64_t *>(b->ws->scan_tmp.p);
    for (int attempt = 0; attempt < 6; attempt++) {
        const DevBatch d = make_devbatch(b);
        if (attempt > 0 || !small) launch_reset_ctl(d.ctl, st);
        launch_lookup(d, set, ix, rescue ? 2 : 1, st);
        launch_hits(d, ix, rescue_cutoff, hard_cutoff, st);
        launch_merge(d, set, st);
        launch_output(d, 0, tmp, b->ws->h_ctl_dev, st);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipStreamSynchronize(st));
        b->ws->tot_nams = b->ws->h_ctl->tot[2];
        unsigned ovf = b->ws->h_ctl->overflow;
        if (!ovf) break;
        if (attempt == 5) throw HipError{hipErrorOutOfMemory, "batch arrays still too small after regrowth"};
        if (ovf & (OVF_HITS | OVF_RHITS | OVF_MERGE)) ovf &= ~(unsigned)OVF_OUT;
        if (ovf & OVF_MERGE) b->ws->merge_scratch = true;
        if ((ovf & OVF_OUT) && b->host_out && host_out_grow(b, b->ws->tot_nams)) ovf &= ~(unsigned)OVF_OUT;
        ensure_pools(b, (ovf & OVF_HITS) ? b->ws->h_ctl->tot[0] + 4096 : 0,
                     (ovf & OVF_RHITS) ? b->ws->h_ctl->tot[1] + 4096 : 0,
                     (ovf & OVF_OUT) ? b->ws->tot_nams + 1024 : 0);
    }
    guard.armed = false;
    b->ran = true;
    note_nams(b);
    return batch_download(b, out);
}

namespace {

// Concurrent per-read calls (the reference's find_nams is re-entrant and
// called once per read from many threads, step2/nam.cu:553-562) are
// combined: a call queues itself; whichever caller finds the context free
// takes every queued call with the same rescue settings and runs them as one
// batch, then hands each caller its reads' results.
struct QrsCall {
    const gis_query_randstrobe *qrs;
    const uint64_t *qoff;
    uint32_t n;
    int rescue;
    uint32_t rcut, hard;
    gis_nam_out *out;
    int rc = GIS_OK;
    bool done = false;
};

int run_combined(gis_ctx *ctx, std::vector<QrsCall *> &calls) {
    // a call on its own needs no joined arrays
    if (calls.size() == 1 && calls[0]->qoff[0] == 0) {
        QrsCall *c = calls[0];
        c->rc = qrs_run(ctx, c->qrs, c->qoff, c->n, c->rescue, c->rcut, c->hard, c->out);
        return c->rc;
    }
    // one batch: the calls' reads back to back
    uint32_t n = 0;
    uint64_t nq = 0;
    for (QrsCall *c : calls) {
        n += c->n;
        nq += c->qoff[c->n] - c->qoff[0];
    }
    std::vector<gis_query_randstrobe> q(nq);
    std::vector<uint64_t> off(n + 1);
    uint64_t at = 0;
    uint32_t r = 0;
    for (QrsCall *c : calls) {
        const uint64_t lo = c->qoff[0], hi = c->qoff[c->n];
        if (hi > lo) std::memcpy(q.data() + at, c->qrs + lo, (hi - lo) * sizeof(gis_query_randstrobe));
        for (uint32_t i = 0; i < c->n; i++) off[r + i] = at + c->qoff[i] - lo;
        at += hi - lo;
        r += c->n;
    }
    off[n] = at;
    std::vector<uint64_t> noff(n + 1);
    std::vector<float> frac(n);
    std::vector<uint8_t> flags(n);
    std::vector<gis_nam> nams(16 + 4ull * at);
    int rc;
    for (;;) {
        gis_nam_out o{noff.data(), nams.data(), nams.size(), frac.data(), flags.data(), 0};
        rc = qrs_run(ctx, q.data(), off.data(), n, calls[0]->rescue, calls[0]->rcut, calls[0]->hard, &o);
        if (rc == GIS_ERR_CAPACITY && o.n_nams > nams.size()) {
            nams.resize(o.n_nams);
            continue;
        }
        break;
    }
    r = 0;
    for (QrsCall *c : calls) {
        if (rc != GIS_OK) {
            c->rc = rc;
            r += c->n;
            continue;
        }
        gis_nam_out *o = c->out;
        const uint64_t a = noff[r], e = noff[r + c->n];
        o->n_nams = e - a;
        if (o->nam_capacity < e - a || (e > a && !o->nams)) {
            c->rc = GIS_ERR_CAPACITY;
        } else {
            if (o->nam_offsets)
                for (uint32_t i = 0; i <= c->n; i++) o->nam_offsets[i] = noff[r + i] - a;
            if (e > a) std::memcpy(o->nams, nams.data() + a, (e - a) * sizeof(gis_nam));
            if (o->nonrepetitive_fraction && c->n) std::memcpy(o->nonrepetitive_fraction, frac.data() + r, 4ull * c->n);
            if (o->flags && c->n) std::memcpy(o->flags, flags.data() + r, c->n);
            c->rc = GIS_OK;
        }
        r += c->n;
    }
    return rc;
}

}  // namespace

extern "C" int gis_find_nams_qrs(gis_ctx *ctx, const gis_query_randstrobe *qrs,
                                 const uint64_t *query_offsets, uint32_t n_queries, int rescue,
                                 uint32_t rescue_cutoff, uint32_t hard_cutoff, gis_nam_out *out) {
    if (!ctx) return GIS_ERR_BAD_PARAMETER;
    if (!query_offsets || !out) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null argument");
    if (n_queries && !qrs && query_offsets[n_queries] > query_offsets[0])
        return fail(ctx, GIS_ERR_BAD_PARAMETER, "null query randstrobes");
    for (uint64_t i = query_offsets[0]; n_queries && i < query_offsets[n_queries]; i++) {
        if (qrs[i].end > GIS_MAX_READ_LEN) return fail(ctx, GIS_ERR_BAD_PARAMETER, "query end too large");
        if (qrs[i].start > qrs[i].end) return fail(ctx, GIS_ERR_BAD_PARAMETER, "query start after its end");
    }
    QrsCall me{qrs, query_offsets, n_queries, rescue ? 1 : 0, rescue_cutoff, hard_cutoff, out};
    std::unique_lock<std::mutex> l(ctx->comb_mu);
    ctx->comb_queue.push_back(&me);
    while (!me.done) {
        if (ctx->comb_busy) {
            ctx->comb_cv.wait(l);
            continue;
        }
        // this caller runs the queued calls that share its rescue settings
        ctx->comb_busy = true;
        std::vector<QrsCall *> take, keep;
        for (void *v : ctx->comb_queue) {
            QrsCall *c = static_cast<QrsCall *>(v);
            const bool same = c->rescue == me.rescue && (!me.rescue || (c->rcut == me.rcut && c->hard == me.hard));
            (same ? take : keep).push_back(c);
        }
        ctx->comb_queue.assign(keep.begin(), keep.end());
        l.unlock();
        int rc = GIS_OK;
        {
            std::lock_guard<std::recursive_mutex> lk(ctx->mu);
            try {
                HIP_CHECK(hipSetDevice(ctx->device));
                rc = run_combined(ctx, take);
            } catch (const HipError &e) {
                rc = hip_fail(ctx, e);
            } catch (const std::bad_alloc &) {
                rc = fail(ctx, GIS_ERR_NOMEM, "host allocation failed");
            }
        }
        l.lock();
        for (QrsCall *c : take) {
            if (rc != GIS_OK) c->rc = rc;
            c->done = true;
        }
        ctx->comb_busy = false;
        ctx->comb_cv.notify_all();
    }
    return me.rc;
}

// ---------------- device-resident batches ----------------

static const char *const IN_FLIGHT_MSG = "a launched run on this batch's workspace was not waited for";

extern "C" int gis_batch_create(gis_ctx *ctx, uint32_t max_reads, uint64_t max_bases, gis_batch **out) {
    API_BEGIN(ctx)
    if (!out) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null output");
    gis_batch *b = batch_new(ctx, nullptr);
    ensure_input_arrays(b, max_reads);
    ensure_read_arrays(b, max_reads);
    ensure<char>(b->seqs, max_bases + SEQ_PAD);
    *out = b;
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_batch_create_async(gis_ctx *ctx, uint32_t max_reads, uint64_t max_bases, gis_batch **out) {
    API_BEGIN(ctx)
    if (!out) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null output");
    gis_batch *b = batch_new_stream(ctx);
    try {
        ensure_input_arrays(b, max_reads);
        ensure_read_arrays(b, max_reads);
        ensure<char>(b->seqs, max_bases + SEQ_PAD);
    } catch (...) {
        batch_free(b);
        throw;
    }
    *out = b;
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_batch_create_shared(gis_ctx *ctx, uint32_t max_reads, uint64_t max_bases,
                                       gis_batch *share_with, gis_batch **out) {
    API_BEGIN(ctx)
    if (!out || !share_with) return fail(ctx, GIS_ERR_BAD_PARAMETER, "null argument");
    if (share_with->ctx != ctx) return fail(ctx, GIS_ERR_BAD_PARAMETER, "the batch belongs to another context");
    gis_batch *b = batch_new(ctx, share_with->ws);
    b->stream = share_with->stream;
    ensure_input_arrays(b, max_reads);
    ensure<char>(b->seqs, max_bases + SEQ_PAD);
    *out = b;
    return GIS_OK;
    API_END(ctx)
}

extern "C" void gis_batch_destroy(gis_batch *b) {
    if (!b) return;
    gis_ctx *ctx = b->ctx;
    std::lock_guard<std::recursive_mutex> lk(ctx->mu);
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(b->stream);
    batch_free(b);
}

extern "C" int gis_batch_upload(gis_batch *b, const char *seqs, const uint64_t *offsets,
                                const uint32_t *lens, uint32_t n_reads) {
    if (!b) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    if (b->ws->in_flight) return fail(ctx, GIS_ERR_STATE, IN_FLIGHT_MSG);
    return batch_upload(b, seqs, offsets, lens, n_reads, false);
    API_END(ctx)
}

extern "C" int gis_batch_run(gis_batch *b, const gis_map_options *opt) {
    if (!b) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    if (!ctx->ix.loaded) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    if (b->ws->in_flight) return fail(ctx, GIS_ERR_STATE, IN_FLIGHT_MSG);
    batch_run(b, opts_or_default(opt), 0, STOP_NONE);
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_batch_launch(gis_batch *b, const gis_map_options *opt) {
    if (!b) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    if (!ctx->ix.loaded) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    if (b->ws->in_flight) return fail(ctx, GIS_ERR_STATE, IN_FLIGHT_MSG);
    b->pending_opt = opts_or_default(opt);
    if (ctx->launched == 0) {  // a burst starts
        ctx->burst = true;
        ctx->turn_st = nullptr;
    }
    batch_launch(b, run_opts(b, b->pending_opt, 0, STOP_NONE), ctx->burst);
    b->ws->in_flight = b;
    ctx->launched++;
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_batch_wait(gis_batch *b) {
    if (!b) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    if (b->ws->in_flight != b) return fail(ctx, GIS_ERR_STATE, "no launched run of this batch to wait for");
    // released first: after an error the workspace takes runs again
    b->ws->in_flight = nullptr;
    ctx->launched--;
    ctx->burst = false;
    batch_complete(b, run_opts(b, b->pending_opt, 0, STOP_NONE));
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_batch_download(gis_batch *b, gis_nam_out *out) {
    if (!b) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    return batch_download(b, out);
    API_END(ctx)
}

extern "C" int gis_batch_nam_count(gis_batch *b, uint64_t *n_nams) {
    if (!b || !n_nams) return GIS_ERR_BAD_PARAMETER;
    if (b->ws->owner != b || b->ws->in_flight) return GIS_ERR_STATE;
    *n_nams = b->ws->tot_nams;
    return GIS_OK;
}

extern "C" int gis_batch_stage_times(gis_batch *b, double *ms, int cap, int *n, char *names, int names_cap) {
    if (!b) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    if (b->ws->in_flight) return fail(ctx, GIS_ERR_STATE, IN_FLIGHT_MSG);
    if (b->last_graph)
        return fail(ctx, GIS_ERR_STATE, "stage times need a run with GIS_RUN_NO_GRAPH (graph replays carry no events)");
    std::string nm;
    int k = 0;
    for (int i = 1; i < b->n_ev && k < cap; i++, k++) {
        float t = 0;
        HIP_CHECK(hipEventElapsedTime(&t, b->ev[i - 1], b->ev[i]));
        if (ms) ms[k] = t;
        if (!nm.empty()) nm += ",";
        nm += b->ev_names[i];
    }
    if (n) *n = k;
    if (names && names_cap > 0) std::snprintf(names, (size_t)names_cap, "%s", nm.c_str());
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_batch_lookup_bytes(gis_batch *b, uint64_t *bytes, uint64_t *n_lookups) {
    if (!b) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    if (b->ws->owner != b) return fail(ctx, GIS_ERR_STATE, "another batch ran on the shared workspace since");
    if (!b->ran) return fail(ctx, GIS_ERR_STATE, "batch has not been run");
    if (b->last_mode != GIS_MODE_PLAIN) return fail(ctx, GIS_ERR_STATE, "lookup bytes are counted by the per-stage path");
    const uint32_t n = b->n_reads;
    std::vector<uint32_t> by(n), cnt(n);
    if (n) {
        HIP_CHECK(hipMemcpy(by.data(), b->ws->lk_bytes.p, 4ull * n, hipMemcpyDeviceToHost));
        HIP_CHECK(hipMemcpy(cnt.data(), b->ws->rs_cnt.p, 4ull * n, hipMemcpyDeviceToHost));
    }
    uint64_t tb = 0, tq = 0;
    for (uint32_t r = 0; r < n; r++) {
        tb += by[r];
        tq += cnt[r];
    }
    if (bytes) *bytes = tb;
    if (n_lookups) *n_lookups = tq;
    return GIS_OK;
    API_END(ctx)
}

extern "C" int gis_batch_lookup_streams(gis_batch *b, uint64_t *stream_bytes) {
    if (!b || !stream_bytes) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    if (b->ws->owner != b) return fail(ctx, GIS_ERR_STATE, "another batch ran on the shared workspace since");
    if (!b->ran) return fail(ctx, GIS_ERR_STATE, "batch has not been run");
    if (b->last_mode != GIS_MODE_PLAIN) return fail(ctx, GIS_ERR_STATE, "lookup bytes are counted by the per-stage path");
    const uint32_t n = b->n_reads;
    std::vector<uint32_t> sb(n);
    if (n) HIP_CHECK(hipMemcpy(sb.data(), b->ws->lk_stream.p, 4ull * n, hipMemcpyDeviceToHost));
    uint64_t t = 0;
    for (uint32_t r = 0; r < n; r++) t += sb[r];
    *stream_bytes = t;
    return GIS_OK;
    API_END(ctx)
}

// ---------------- autotuner of the fused form ----------------

extern "C" int gis_batch_autotune(gis_batch *b, const gis_map_options *opt, gis_fused_config *best,
                                  double *best_ms, uint32_t *n_tried) {
    if (!b) return GIS_ERR_BAD_PARAMETER;
    gis_ctx *ctx = b->ctx;
    API_BEGIN(ctx)
    if (!ctx->ix.loaded) return fail(ctx, GIS_ERR_STATE, "no index loaded");
    if (b->n_reads == 0) return fail(ctx, GIS_ERR_STATE, "no reads uploaded");
    if (b->ws->in_flight) return fail(ctx, GIS_ERR_STATE, IN_FLIGHT_MSG);
    gis_map_options o = opts_or_default(opt);
    o.mode = GIS_MODE_FUSED;
    o.flags |= GIS_RUN_NO_GRAPH;
    // candidates: waves per block x length split x queue discipline
    struct Q { int queue, chunk, bpc; };
    const Q queues[] = {{0, 0, 0}, {0, 0, 4}, {0, 0, 8}, {1, 4, 4}, {1, 4, 8}, {1, 16, 8}, {1, 64, 4}};
    std::vector<gis_fused_config> cands;
    for (int w : {2, 4, 8})
        for (int split : {0, 1})
            for (const Q &q : queues) cands.push_back(gis_fused_config{w, split, q.queue, q.chunk, q.bpc});
    const gis_fused_config saved = ctx->fcfg;
    double bt = 1e300;
    gis_fused_config bc = saved;
    try {
        for (const gis_fused_config &c : cands) {
            ctx->fcfg = c;
            batch_run(b, o, 0, STOP_NONE);  // first launch of the variant; pools sized
            double t = 1e300;
            for (int rep = 0; rep < 3; rep++) {
                const auto t0 = std::chrono::steady_clock::now();
                batch_run(b, o, 0, STOP_NONE);
                const double ms =
                    std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
                t = std::min(t, ms);
            }
            if (t < bt) {
                bt = t;
                bc = c;
            }
        }
    } catch (...) {
        ctx->fcfg = saved;
        throw;
    }
    ctx->fcfg = bc;
    if (best) *best = bc;
    if (best_ms) *best_ms = bt;
    if (n_tried) *n_tried = (uint32_t)cands.size();
    return GIS_OK;
    API_END(ctx)
}
