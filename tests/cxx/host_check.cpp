// Drives the C ABI with the runtime's calls watched: this program defines some of
// the HIP entry points that libgis.so calls, counts them, and hands them on, or
// fails an allocation as a device without room would. (No GPU memory is ever
// exhausted for it.)
//
// usage: host_check <case>; exit status 0 if the case holds
#include <dlfcn.h>

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
std::map<void *, uint64_t> g_copy, g_sync;  // streams: when last copied in on, when last waited for
uint64_t g_clock = 0;

}  // namespace

extern "C" int hipMalloc(void **p, size_t n) {
    static const auto f = real<int (*)(void **, size_t)>("hipMalloc");
    bool fail;
    {
        std::lock_guard<std::mutex> l(g_mu);
        fail = g_no_room;
    }
    if (!fail) return f(p, n);
    std::this_thread::sleep_for(std::chrono::milliseconds(300));
    *p = nullptr;
    return 2;
}

extern "C" int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
    static const auto f = real<int (*)(void *, const void *, size_t, int, void *)>("hipMemcpyAsync");
    {
        std::lock_guard<std::mutex> l(g_mu);
        if (kind == 1) g_copy[st] = ++g_clock;
    }
    return f(d, s, n, kind, st);
}

extern "C" int hipStreamSynchronize(void *st) {
    static const auto f = real<int (*)(void *)>("hipStreamSynchronize");
    const int e = f(st);
    std::lock_guard<std::mutex> l(g_mu);
    g_sync[st] = ++g_clock;
    return e;
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

static Genome genome(uint64_t n, uint32_t contigs, uint64_t seed) {
    gis_genome_spec s{};
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

static Reads reads(const Genome &g, uint32_t n, uint32_t len, uint64_t seed) {
    gis_read_spec s{};
    s.n_reads = n;
    s.lengths[0] = len;
    s.weights[0] = 1;
    s.n_lengths = 1;
    s.sub_rate = 0.005;
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

int main(int argc, char **argv) {
    const struct {
        const char *name;
        void (*run)();
    } cases[] = {{"pinned_ranges", pinned_ranges}, {"stream_failure", stream_failure}};
    for (const auto &c : cases)
        if (argc == 2 && !std::strcmp(argv[1], c.name)) {
            c.run();
            std::printf("%s holds\n", c.name);
            return 0;
        }
    std::fprintf(stderr, "usage: host_check <case>\n");
    return 2;
}
