// Drives the C ABI with the runtime's calls watched: this program defines some of
// the HIP entry points that libgis.so calls, counts them, and hands them on, or
// fails an allocation as a device without room would. (No GPU memory is ever
// exhausted for it.)
//
// usage: host_check <case>; exit status 0 if the case holds
#include <dlfcn.h>
#include <sys/resource.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/gis.h"

namespace gis {
bool pinned_range(const void *p, size_t bytes);  // csrc/host_copy.h
}

#define EXPECT(x)                                                          \
    do {                                                                   \
        if (!(x)) {                                                        \
            std::fprintf(stderr, "%s:%d: not so: %s\n", __FILE__, __LINE__, #x); \
            std::exit(1);                                                  \
        }                                                                  \
    } while (0)

// ---------------- the watched calls ----------------
// (hipError_t is an int here: 0 success, 2 out of memory)

namespace {

template <typename F>
F real(const char *name) {
    void *f = dlsym(RTLD_NEXT, name);
    EXPECT(f);
    return reinterpret_cast<F>(f);
}

std::mutex g_mu;
bool g_no_room = false;                    // hipMalloc fails, and says so late
uint64_t g_limit = UINT64_MAX;             // device bytes there are to allocate
uint64_t g_live = 0, g_peak = 0;           // allocated now, and at most
std::map<void *, uint64_t> g_blocks;
std::map<void *, uint64_t> g_copy, g_sync;  // streams: when last copied in on, when last waited for
uint64_t g_clock = 0;
std::atomic<uint64_t> g_launches{0}, g_graphs{0}, g_made{0};  // kernels and graphs, graphs alone, graphs made

std::atomic<int> g_stall{0};  // milliseconds that the next wait for an event takes longer

struct Dim3 {
    uint32_t x, y, z;
};

// host arrays of copies in to the device that their streams were not waited for since
struct Src {
    const char *p;
    size_t n;
    void *st;
};
constexpr int MAX_SRC = 4096;
Src g_src[MAX_SRC];
int g_n_src = 0;
std::mutex g_src_mu;             // (not g_mu, under which memory is freed)
std::atomic<int> g_freed{0};     // those freed all the same

}  // namespace

void operator delete(void *p) noexcept {
    const char *c = static_cast<const char *>(p);
    if (c) {
        std::lock_guard<std::mutex> l(g_src_mu);
        for (int i = 0; i < g_n_src; i++) g_freed += g_src[i].p == c;
    }
    std::free(p);
}
void operator delete(void *p, size_t) noexcept { operator delete(p); }

extern "C" int hipMalloc(void **p, size_t n) {
    static const auto f = real<int (*)(void **, size_t)>("hipMalloc");
    std::unique_lock<std::mutex> l(g_mu);
    if (g_no_room || g_limit - std::min(g_limit, g_live) < n) {
        const bool late = g_no_room;
        l.unlock();
        if (late) std::this_thread::sleep_for(std::chrono::milliseconds(300));
        *p = nullptr;
        return 2;
    }
    const int e = f(p, n);
    if (e) return e;
    g_blocks[*p] = n;
    g_live += n;
    g_peak = std::max(g_peak, g_live);
    return e;
}

extern "C" int hipFree(void *p) {
    static const auto f = real<int (*)(void *)>("hipFree");
    {
        std::lock_guard<std::mutex> l(g_mu);
        const auto b = g_blocks.find(p);
        if (b != g_blocks.end()) {
            g_live -= b->second;
            g_blocks.erase(b);
        }
    }
    return f(p);
}

extern "C" int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
    static const auto f = real<int (*)(void *, const void *, size_t, int, void *)>("hipMemcpyAsync");
    {
        std::lock_guard<std::mutex> l(g_mu);
        if (kind == 1) g_copy[st] = ++g_clock;
    }
    if (kind == 1) {
        std::lock_guard<std::mutex> l(g_src_mu);
        if (g_n_src < MAX_SRC) g_src[g_n_src++] = {static_cast<const char *>(s), n, st};
    }
    return f(d, s, n, kind, st);
}

extern "C" int hipStreamSynchronize(void *st) {
    static const auto f = real<int (*)(void *)>("hipStreamSynchronize");
    const int e = f(st);
    {
        std::lock_guard<std::mutex> l(g_src_mu);
        g_n_src = (int)(std::remove_if(g_src, g_src + g_n_src, [&](const Src &x) { return x.st == st; }) - g_src);
    }
    std::lock_guard<std::mutex> l(g_mu);
    g_sync[st] = ++g_clock;
    return e;
}

extern "C" int hipLaunchKernel(const void *k, Dim3 grid, Dim3 block, void **args, size_t lds, void *st) {
    static const auto f = real<int (*)(const void *, Dim3, Dim3, void **, size_t, void *)>("hipLaunchKernel");
    g_launches++;
    return f(k, grid, block, args, lds, st);
}

extern "C" int hipGraphLaunch(void *exec, void *st) {
    static const auto f = real<int (*)(void *, void *)>("hipGraphLaunch");
    g_launches++;
    g_graphs++;
    return f(exec, st);
}

extern "C" int hipGraphInstantiate(void **exec, void *graph, void **node, char *log, size_t n) {
    static const auto f = real<int (*)(void **, void *, void **, char *, size_t)>("hipGraphInstantiate");
    g_made++;
    return f(exec, graph, node, log, n);
}

extern "C" int hipEventSynchronize(void *ev) {
    static const auto f = real<int (*)(void *)>("hipEventSynchronize");
    std::this_thread::sleep_for(std::chrono::milliseconds(g_stall.exchange(0)));
    return f(ev);
}

// ---------------- inputs ----------------

struct Genome {
    std::vector<char> seq;
    std::vector<uint64_t> lens;
    std::vector<const char *> at() const {
        std::vector<const char *> a;
        const char *p = seq.data();
        for (uint64_t n : lens) a.push_back(p), p += n;
        return a;
    }
};

static Genome genome(uint64_t n, uint32_t contigs, uint64_t seed, double repeats = 0) {
    gis_genome_spec s{};
    s.repeat_fraction = repeats;
    s.n_families = 4;
    s.family_min_len = 600;
    s.family_max_len = 900;
    s.copies_min = 150;
    s.copies_max = 250;
    s.total_length = n;
    s.n_contigs = contigs;
    s.gc = 0.45;
    s.seed = seed;
    Genome g;
    g.seq.resize(n);
    g.lens.resize(contigs);
    EXPECT(gis_synth_genome(&s, g.seq.data(), g.lens.data()) == GIS_OK);
    return g;
}

struct Reads {
    std::vector<char> seqs;
    std::vector<uint64_t> offs;
    std::vector<uint32_t> lens;
    uint32_t n() const { return (uint32_t)lens.size(); }
    void add(const Reads &o) {
        for (uint64_t x : o.offs) offs.push_back(x + seqs.size());
        lens.insert(lens.end(), o.lens.begin(), o.lens.end());
        seqs.insert(seqs.end(), o.seqs.begin(), o.seqs.end());
    }
};

static Reads reads(const Genome &g, uint32_t n, uint32_t len, uint64_t seed, double errors = 0.005) {
    gis_read_spec s{};
    s.n_reads = n;
    s.lengths[0] = len;
    s.weights[0] = 1;
    s.n_lengths = 1;
    s.sub_rate = errors;
    s.indel_rate = errors / 5;
    s.rc_fraction = 0.5;
    s.seed = seed;
    Reads r;
    r.seqs.resize((size_t)n * len);
    r.offs.resize(n);
    r.lens.resize(n);
    std::vector<uint32_t> c(n), p(n);
    std::vector<uint8_t> rc(n);
    EXPECT(gis_synth_reads(&s, g.seq.data(), g.lens.data(), (uint32_t)g.lens.size(), r.seqs.data(), r.offs.data(),
                           r.lens.data(), c.data(), p.data(), rc.data()) == GIS_OK);
    return r;
}

static gis_params params(int read_length) {
    gis_params p;
    EXPECT(gis_params_from_read_length(read_length, GIS_DEFAULT, GIS_DEFAULT, GIS_DEFAULT, GIS_DEFAULT, GIS_DEFAULT,
                                       GIS_DEFAULT, &p) == GIS_OK);
    return p;
}

static int build(gis_ctx *ctx, const Genome &g, int bits = -1) {
    const gis_params p = params(150);
    return gis_index_build(ctx, g.at().data(), g.lens.data(), (uint32_t)g.lens.size(), &p, bits, 0.0002f, 1);
}

static gis_ctx *context() {
    gis_ctx *ctx = nullptr;
    EXPECT(gis_ctx_create(0, &ctx) == GIS_OK);
    return ctx;
}

// ---------------- cases ----------------

// a kernel may write an array only where it is pinned to its last byte
static void pinned_ranges() {
    constexpr size_t N = 1 << 20, PAST = 4 << 20;
    void *v = nullptr;
    EXPECT(gis_host_alloc(N, &v) == GIS_OK);
    char *p = static_cast<char *>(v);
    EXPECT(gis::pinned_range(p, N) && gis::pinned_range(p + 16, N - 16) && gis::pinned_range(p + N - 1, 1));
    EXPECT(!gis::pinned_range(p, N + PAST) && !gis::pinned_range(p + N - 1, 1 + PAST));
    std::vector<char> heap(N);
    EXPECT(!gis::pinned_range(heap.data(), N) && !gis::pinned_range(heap.data(), 1));
    gis_host_free(v);
}

// a lane of a stream that fails takes the others with it: they have staged their
// batches by then, and wait for those copies before the call returns
static void stream_failure() {
    const Genome g = genome(200000, 1, 1);
    gis_ctx *ctx = context();
    EXPECT(build(ctx, g) == GIS_OK);
    const uint32_t per = 256;
    Reads r = reads(g, per, 2000, 2);  // the first batch: its run needs scratch for long reads
    r.add(reads(g, 3 * per, 150, 3));
    std::vector<uint64_t> off(r.n() + 1);
    std::vector<gis_nam> nams(64 * (size_t)r.n());
    gis_nam_out o{off.data(), nams.data(), nams.size(), nullptr, nullptr, 0};
    const auto run = [&](uint32_t from) {
        return gis_find_nams_stream(ctx, r.seqs.data(), r.offs.data() + from, r.lens.data() + from, r.n() - from, per, 4,
                                    nullptr, &o, nullptr);
    };
    // the short ones in every lane once
    Reads s = reads(g, 4 * per, 150, 4);
    EXPECT(gis_find_nams_stream(ctx, s.seqs.data(), s.offs.data(), s.lens.data(), s.n(), per, 4, nullptr, &o, nullptr) ==
           GIS_OK);
    {
        std::lock_guard<std::mutex> l(g_mu);
        g_no_room = true;
        g_copy.clear();
    }
    EXPECT(run(0) == GIS_ERR_HIP);
    {
        std::lock_guard<std::mutex> l(g_mu);
        g_no_room = false;
        EXPECT(g_copy.size() >= 3);  // (the other lanes' streams)
        for (const auto &c : g_copy) EXPECT(g_sync[c.first] > c.second);
    }
    EXPECT(run(0) == GIS_OK);
    gis_ctx_destroy(ctx);
}

// A table that fits an empty device fits one that holds another: replacing it takes
// no more memory than loading it first does, whatever was kept of the one before.
// A load that cannot fit leaves nothing allocated, and the next one works.
static void replace_index() {
    const Genome small = genome(300000, 2, 5), large = genome(3000000, 2, 6);
    const std::string path = std::string(std::getenv("TMPDIR") ? std::getenv("TMPDIR") : "/tmp") + "/host_check_" +
                             std::to_string((long)std::chrono::steady_clock::now().time_since_epoch().count()) + ".sti";
    const int BITS = 18, BITS_BEFORE = 22;
    // the table three ways
    std::vector<gis_ref_randstrobe> rs;
    std::vector<uint64_t> starts((1ull << BITS) + 1);
    gis_index_info want{};
    {
        gis_ctx *ctx = context();
        EXPECT(build(ctx, large, BITS) == GIS_OK && gis_index_info_get(ctx, &want) == GIS_OK);
        rs.resize(want.n_randstrobes);
        EXPECT(gis_index_download(ctx, rs.data(), starts.data()) == GIS_OK);
        EXPECT(gis_index_write_sti(ctx, path.c_str()) == GIS_OK);
        gis_ctx_destroy(ctx);
    }
    const auto load = [&](gis_ctx *ctx, int how) {
        if (how == 0) return build(ctx, large, BITS);
        if (how == 1)
            return gis_index_upload(ctx, rs.data(), rs.size(), starts.data(), BITS, want.filter_cutoff, &want.params);
        return gis_index_read_sti(ctx, path.c_str(), nullptr);
    };
    const auto same = [&](gis_ctx *ctx) {
        std::vector<gis_ref_randstrobe> r(rs.size());
        std::vector<uint64_t> s(starts.size());
        gis_index_info i{};
        EXPECT(gis_index_info_get(ctx, &i) == GIS_OK && i.n_randstrobes == rs.size() && i.bits == BITS);
        EXPECT(gis_index_download(ctx, r.data(), s.data()) == GIS_OK);
        EXPECT(!std::memcmp(r.data(), rs.data(), rs.size() * sizeof rs[0]) && s == starts);
    };
    for (int how = 0; how < 3; how++) {
        const uint64_t none = g_live;
        gis_ctx *ctx = context();
        g_peak = g_live;
        EXPECT(load(ctx, how) == GIS_OK);
        const uint64_t alone = g_peak;
        gis_ctx_destroy(ctx);
        EXPECT(g_live == none);
        for (int before = 0; before < 2; before++) {  // many buckets; many records
            ctx = context();
            EXPECT((before ? build(ctx, large, BITS - 2) : build(ctx, small, BITS_BEFORE)) == GIS_OK);
            g_limit = alone;
            EXPECT(load(ctx, how) == GIS_OK);
            same(ctx);
            EXPECT(g_live <= alone);
            // too little for more buckets, and then for any load
            g_limit = none + (1 << 20);
            EXPECT(build(ctx, large, BITS_BEFORE + 1) == GIS_ERR_HIP);
            EXPECT(g_live == none);
            EXPECT(load(ctx, how) == GIS_ERR_HIP);
            EXPECT(g_live == none);
            EXPECT(gis_index_info_get(ctx, &want) == GIS_ERR_STATE);
            g_limit = UINT64_MAX;
            EXPECT(load(ctx, how) == GIS_OK);
            same(ctx);
            gis_ctx_destroy(ctx);
            EXPECT(g_live == none);
        }
    }
    // a build whose own memory stays with the context when there is room, and goes
    // before the bucket lines (here most of the table) need it
    const uint64_t none = g_live;
    gis_ctx *ctx = context();
    EXPECT(build(ctx, small, BITS_BEFORE) == GIS_OK && gis_index_info_get(ctx, &want) == GIS_OK);
    gis_ctx_destroy(ctx);
    ctx = context();
    g_limit = none + want.n_randstrobes * 16 + ((1ull << BITS_BEFORE) + 1) * 8 + (128ull << BITS_BEFORE) + (1 << 20);
    EXPECT(build(ctx, small, BITS_BEFORE) == GIS_OK);
    gis_ctx_destroy(ctx);
    g_limit = UINT64_MAX;
    std::remove(path.c_str());
}

// Seeding a reference that finds no memory, at any of its arrays, frees no host array
// that a copy to the device may still read.
static void build_failure() {
    const Genome g = genome(3000000, 40, 12);
    uint64_t total = 0, n = 0;
    for (uint64_t x : g.lens) total += x;
    const gis_params p = params(150);
    gis_ctx *ctx = context();
    const auto at = g.at();
    int failed = 0, rc = GIS_ERR_HIP;
    std::vector<gis_ref_randstrobe> out(total);
    for (g_limit = g_live + (1 << 16); rc; g_limit += 1 << 19) {
        g_freed = 0;
        rc = gis_reference_randstrobes(ctx, at.data(), g.lens.data(), (uint32_t)g.lens.size(), &p, out.data(), total,
                                       &n);
        EXPECT(rc == GIS_OK || rc == GIS_ERR_HIP);
        EXPECT(g_freed == 0);
        failed += rc != GIS_OK;
    }
    EXPECT(failed > 8 && n > 0);
    g_limit = UINT64_MAX;
    gis_ctx_destroy(ctx);
}

// an index's device bytes are those of its table, whatever was resident before it
static void index_bytes() {
    const Genome small = genome(100000, 1, 7), large = genome(1000000, 1, 8);
    gis_ctx *ctx = context();
    EXPECT(build(ctx, large, 14) == GIS_OK);
    for (int bits : {14, 13, 16}) {
        gis_index_info i{};
        EXPECT(build(ctx, small, bits) == GIS_OK && gis_index_info_get(ctx, &i) == GIS_OK);
        EXPECT(i.device_bytes == i.n_randstrobes * 16 + ((1ull << bits) + 1) * 8 + (128ull << bits));
    }
    gis_ctx_destroy(ctx);
}

// the device memory of a pair step follows its lists, not max_tries
static void pairs_memory() {
    gis_ctx *ctx = context();
    const uint32_t n = 100000;
    std::vector<uint64_t> off(2 * n + 1);
    std::vector<gis_nam> nams(2 * n);
    for (uint32_t r = 0; r < 2 * n; r++) {
        off[r + 1] = r + 1;
        gis_nam &x = nams[r];
        x = gis_nam{};
        x.query_end = 50;
        x.ref_start = 1000 + r % n + (r < n ? 0 : 200);
        x.ref_end = x.ref_start + 50;
        x.n_hits = 3;
        x.score = 30;
        x.is_rc = r >= n;
    }
    gis_pair_params p;
    gis_pair_params_default(&p);
    p.max_tries = 256;
    p.flags = GIS_PAIRS_JOINT;
    std::vector<gis_nam_pair> joint(n);
    std::vector<uint64_t> joff(n + 1);
    gis_pair_out o{};
    o.joint = joint.data();
    o.joint_capacity = n;
    o.joint_offsets = joff.data();
    const uint64_t before = g_live;
    EXPECT(gis_pairs_from_nams(ctx, off.data(), nams.data(), n, &p, &o) == GIS_OK);
    EXPECT(g_live - before < 100u << 20);
    EXPECT(o.n_joint == n && joff[n] == n);
    for (const gis_nam_pair &e : joint) EXPECT(e.score == 6 && e.i1 == 0 && e.i2 == 0);
    gis_ctx_destroy(ctx);
}

// A call on NAM lists that finds no memory once their copies are in flight waits for
// them before it returns the caller's arrays.
static void pairs_failure() {
    const uint32_t n = 2000, each = 20;
    std::vector<uint64_t> off(2 * n + 1);
    std::vector<gis_nam> nams(2 * n * each);
    for (uint32_t r = 0; r < 2 * n; r++) {
        off[r + 1] = (r + 1ull) * each;
        for (uint32_t i = 0; i < each; i++) {
            gis_nam &x = nams[(size_t)r * each + i];
            x = gis_nam{};
            x.query_end = 50;
            x.ref_start = 1000 + 100 * (int)i + (r < n ? 0 : 200);
            x.ref_end = x.ref_start + 50;
            x.n_hits = 3;
            x.score = 30;
            x.is_rc = r >= n;
        }
    }
    gis_pair_params p;
    gis_pair_params_default(&p);
    std::vector<uint8_t> types(n), want(n);
    gis_pair_out o{};
    o.types = want.data();
    gis_ctx *ctx = context();
    EXPECT(gis_pairs_from_nams(ctx, off.data(), nams.data(), n, &p, &o) == GIS_OK);
    gis_ctx_destroy(ctx);
    ctx = context();
    o.types = types.data();
    int failed = 0, rc = GIS_ERR_HIP;
    const uint64_t lists = off.size() * 8 + nams.size() * sizeof(gis_nam);
    for (g_limit = g_live + lists; rc; g_limit += lists / 4) {
        g_copy.clear();
        g_sync.clear();
        rc = gis_pairs_from_nams(ctx, off.data(), nams.data(), n, &p, &o);
        EXPECT(rc == GIS_OK || rc == GIS_ERR_HIP);
        if (rc && !g_copy.empty()) failed++;
        for (const auto &c : g_copy) EXPECT(g_sync.count(c.first) && g_sync[c.first] > c.second);
    }
    EXPECT(failed > 0 && types == want);
    g_limit = UINT64_MAX;
    gis_ctx_destroy(ctx);
}

struct Nams {
    std::vector<uint64_t> off;
    std::vector<gis_nam> nams;
    std::vector<float> frac;
    std::vector<uint8_t> flags;
    gis_nam_out o{};
    Nams(uint32_t n, uint64_t cap) : off(n + 1), nams(cap), frac(n), flags(n) {
        o = gis_nam_out{off.data(), nams.data(), cap, frac.data(), flags.data(), 0};
    }
    bool operator==(const Nams &x) const {
        return o.n_nams == x.o.n_nams && off == x.off && frac == x.frac && flags == x.flags &&
               !std::memcmp(nams.data(), x.nams.data(), o.n_nams * sizeof(gis_nam));
    }
};

// A small call of reads with many NAMs runs once, like any other, when the calls
// before it were like it: more NAMs than pinned room for them at first (100 reads of
// 4000 bp), and more than go that way at all (reads of a repeat).
static void dense_calls() {
    const Genome quiet = genome(1000000, 1, 9), rich = genome(1000000, 1, 10, 0.5);
    for (int kind = 0; kind < 3; kind++) {
        const Genome &g = kind < 2 ? quiet : rich;
        gis_ctx *ctx = context();
        EXPECT(build(ctx, g) == GIS_OK);
        const Reads r = kind == 0 ? reads(g, 100, 150, 11) : kind == 1 ? reads(g, 100, 4000, 11, 0.05) : reads(g, 2500, 300, 11);
        const uint32_t n = r.n();
        // by a resident batch
        gis_batch *b = nullptr;
        EXPECT(gis_batch_create(ctx, n, r.seqs.size(), &b) == GIS_OK);
        EXPECT(gis_batch_upload(b, r.seqs.data(), r.offs.data(), r.lens.data(), n) == GIS_OK);
        EXPECT(gis_batch_run(b, nullptr) == GIS_OK);
        uint64_t total = 0;
        EXPECT(gis_batch_nam_count(b, &total) == GIS_OK);
        Nams want(n, total);
        EXPECT(gis_batch_download(b, &want.o) == GIS_OK);
        gis_batch_destroy(b);
        EXPECT(kind == 0 ? total < 16 * n : kind == 1 ? total > 16 * n + 1024 : total > (4u << 20) / sizeof(gis_nam));
        // host calls
        for (int call = 0; call < 5; call++) {
            Nams got(n, total);
            const uint64_t before = g_launches;
            EXPECT(gis_find_nams_batch(ctx, r.seqs.data(), r.offs.data(), r.lens.data(), n, nullptr, &got.o) == GIS_OK);
            EXPECT(got == want);
            // the inputs and the run's graph; the NAMs of the last kind come by chunks
            if (call > 2) EXPECT(g_launches - before == 2 + (kind < 2 ? 0 : (total * sizeof(gis_nam) - 1) / (1 << 20) + 1));
        }
        // and per query
        std::vector<uint64_t> qoff(n + 1);
        std::vector<gis_query_randstrobe> q(r.seqs.size());
        uint64_t nq = 0;
        EXPECT(gis_randstrobes_batch(ctx, r.seqs.data(), r.offs.data(), r.lens.data(), n, qoff.data(), q.data(), q.size(),
                                     &nq) == GIS_OK);
        uint64_t first = 0;
        for (int call = 0; call < 4; call++) {
            Nams got(n, 2 * total + 1024);
            const uint64_t before = g_launches;
            EXPECT(gis_find_nams_qrs(ctx, q.data(), qoff.data(), n, 0, 0, 0, &got.o) == GIS_OK);
            const uint64_t launches = g_launches - before;
            if (call == 0) first = got.o.n_nams;
            EXPECT(got.o.n_nams == first);
            // (inputs or the reset, lookup, hits, up to four for the merge, two for the output)
            if (call > 0 && kind < 2) EXPECT(launches <= 9);
        }
        gis_ctx_destroy(ctx);
    }
}

// Captured launches hold the addresses of every array they use. The scan's scratch
// grows by tiles of 1024 reads beside arrays that grow by reads, so that a seeding
// call can move it alone: launches captured before are not replayed then.
static void moved_scratch() {
    const Genome g = genome(300000, 1, 12);
    gis_ctx *ctx = context();
    EXPECT(build(ctx, g) == GIS_OK);
    const uint32_t n = 16384, more = 20480;
    const Reads r = reads(g, more, 150, 13);
    // (every kind of room for more than these reads need, half as much again each time)
    Nams got(more, 64ull * more), want(more, 64ull * more);
    const auto call = [&](uint32_t k, Nams &o) {
        return gis_find_nams_batch(ctx, r.seqs.data(), r.offs.data(), r.lens.data(), k, nullptr, &o.o);
    };
    for (uint32_t k : {10240u, 12288u, n, n, n}) EXPECT(call(k, want) == GIS_OK);
    uint64_t graphs = g_graphs;
    EXPECT(call(n, want) == GIS_OK && g_graphs == graphs + 1);
    std::vector<uint64_t> qoff(more + 1);
    std::vector<gis_query_randstrobe> q(128ull * more);
    uint64_t nq = 0;
    EXPECT(gis_randstrobes_batch(ctx, r.seqs.data(), r.offs.data(), r.lens.data(), more, qoff.data(), q.data(), q.size(),
                                 &nq) == GIS_OK);
    graphs = g_graphs;
    EXPECT(call(n, got) == GIS_OK && g_graphs == graphs);
    EXPECT(got == want);
    for (int i = 0; i < 2; i++) EXPECT(call(n, got) == GIS_OK && got == want);
    EXPECT(g_graphs == graphs + 2);
    gis_ctx_destroy(ctx);
}

// A batch keeps the graphs of eight configurations, also where runs in a burst are
// launched in two parts and others whole.
static void graphs_kept() {
    const Genome g = genome(300000, 1, 14);
    gis_ctx *ctx = context();
    EXPECT(build(ctx, g) == GIS_OK);
    const Reads r = reads(g, 16384, 100, 15);  // (as many as take turns)
    gis_batch *b[2];
    for (gis_batch *&x : b) {
        EXPECT(gis_batch_create_async(ctx, r.n(), r.seqs.size(), &x) == GIS_OK);
        EXPECT(gis_batch_upload(x, r.seqs.data(), r.offs.data(), r.lens.data(), r.n()) == GIS_OK);
        EXPECT(gis_batch_run(x, nullptr) == GIS_OK);  // (its arrays have their size)
    }
    uint64_t made[2];
    for (int pass = 0; pass < 2; pass++) {
        const uint64_t before = g_made;
        for (int c = 0; c < 8; c++) {
            gis_map_options o;
            gis_map_options_default(&o);
            o.hard_cutoff = 900 + c;
            for (gis_batch *x : b) EXPECT(gis_batch_launch(x, &o) == GIS_OK);
            for (gis_batch *x : b) EXPECT(gis_batch_wait(x) == GIS_OK);
            for (gis_batch *x : b) EXPECT(gis_batch_run(x, &o) == GIS_OK);
        }
        made[pass] = g_made - before;
    }
    EXPECT(made[0] == 2 * 8 * 3 && made[1] == 0);
    for (gis_batch *x : b) gis_batch_destroy(x);
    gis_ctx_destroy(ctx);
}

// files of uneven reads mapped in turn: 16 configurations of one lane
static void stream_graphs() {
    const Genome g = genome(300000, 1, 16);
    gis_ctx *ctx = context();
    EXPECT(build(ctx, g) == GIS_OK);
    const uint32_t FILES = 4, PER = 1000, BATCHES = 4;
    std::vector<Reads> files;
    for (uint32_t f = 0; f < FILES; f++) {
        Reads r;
        for (uint32_t i = 0; i < BATCHES; i++) {
            const uint32_t longer = 100 + 50 * (f * BATCHES + i);
            r.add(reads(g, PER - longer, 100, 17 + f));
            r.add(reads(g, longer, 300, 18 + f));
        }
        files.push_back(std::move(r));
    }
    Nams out(PER * BATCHES, 400000);
    uint64_t made = 0;
    for (int pass = 0; pass < 4; pass++) {  // (the arrays have their size after the first)
        const uint64_t before = g_made;
        for (const Reads &r : files)
            EXPECT(gis_find_nams_stream(ctx, r.seqs.data(), r.offs.data(), r.lens.data(), r.n(), PER, 1, nullptr, &out.o,
                                        nullptr) == GIS_OK);
        made = g_made - before;
    }
    EXPECT(made == 0);
    gis_ctx_destroy(ctx);
}

// threads of a copy that wait for a chunk the GPU is late with use no CPU time
static void stalled_copy() {
    const Genome g = genome(300000, 1, 16);
    gis_ctx *ctx = context();
    EXPECT(build(ctx, g) == GIS_OK);
    std::vector<uint64_t> keys(4u << 20), pos(keys.size()), want(keys.size());
    for (size_t i = 0; i < keys.size(); i++) keys[i] = i * 0x9e3779b97f4a7c15ull;
    const auto cpu = [&](int stall, std::vector<uint64_t> &out) {
        rusage a, b;
        getrusage(RUSAGE_SELF, &a);
        g_stall = stall;
        EXPECT(gis_lookup_batch(ctx, keys.data(), keys.size(), out.data()) == GIS_OK);
        EXPECT(g_stall == 0);
        getrusage(RUSAGE_SELF, &b);
        const auto ms = [](const timeval &t) { return 1e3 * t.tv_sec + 1e-3 * t.tv_usec; };
        return ms(b.ru_utime) + ms(b.ru_stime) - ms(a.ru_utime) - ms(a.ru_stime);
    };
    double plain = 1e9, late = 1e9;
    cpu(0, want);
    for (int i = 0; i < 3; i++) {
        plain = std::min(plain, cpu(0, pos));
        EXPECT(pos == want);
        std::fill(pos.begin(), pos.end(), 0);
        late = std::min(late, cpu(100, pos));
        EXPECT(pos == want);
    }
    std::printf("CPU %.1f ms, with a chunk 100 ms late %.1f\n", plain, late);
    EXPECT(late - plain < 50);
    gis_ctx_destroy(ctx);
}

int main(int argc, char **argv) {
    const struct {
        const char *name;
        void (*run)();
    } cases[] = {{"pinned_ranges", pinned_ranges}, {"stream_failure", stream_failure}, {"replace_index", replace_index}, {"index_bytes", index_bytes},
                 {"build_failure", build_failure},
                 {"pairs_memory", pairs_memory},
                 {"pairs_failure", pairs_failure},
                 {"dense_calls", dense_calls},
                 {"moved_scratch", moved_scratch},
                 {"graphs_kept", graphs_kept}, {"stream_graphs", stream_graphs}, {"stalled_copy", stalled_copy}};
    for (const auto &c : cases)
        if (argc == 2 && !std::strcmp(argv[1], c.name)) {
            c.run();
            std::printf("%s holds\n", c.name);
            return 0;
        }
    std::fprintf(stderr, "usage: host_check <case>\n");
    return 2;
}
