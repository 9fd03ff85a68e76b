// Drives the C ABI with the runtime's calls watched: this program defines some of
// the HIP entry points that libgis.so calls, counts them, and hands them on, or
// fails an allocation as a device without room would. (No GPU memory is ever
// exhausted for it.)
//
// usage: host_check <case>; exit status 0 if the case holds
#include <dlfcn.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
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

int main(int argc, char **argv) {
    const struct {
        const char *name;
        void (*run)();
    } cases[] = {{"pinned_ranges", pinned_ranges}};
    for (const auto &c : cases)
        if (argc == 2 && !std::strcmp(argv[1], c.name)) {
            c.run();
            std::printf("%s holds\n", c.name);
            return 0;
        }
    std::fprintf(stderr, "usage: host_check <case>\n");
    return 2;
}
