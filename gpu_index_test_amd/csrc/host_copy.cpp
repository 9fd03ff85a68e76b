// Copies between HBM and a caller's arrays (host_copy.h).
#include "host_copy.h"

#include <hsa/hsa.h>
#include <hsa/hsa_ext_amd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "driver_internal.h"
#include "kernels.h"

namespace gis {

namespace {

// pinned memory of the copies: SLOTS chunks in turn
constexpr size_t CHUNK = 1 << 20;
constexpr int SLOTS = 8;
// threads that empty the chunks of a copy of at least THREADS_MIN chunks: the lines
// that the link wrote are in no cache, and one thread reads them at ~22 GB/s, less
// than half the link's rate
constexpr int THREADS = 3;
constexpr uint64_t THREADS_MIN = 4;
// bytes of the arrays that one kernel writes beside a large copy
constexpr uint64_t SMALL_MAX = 8 << 20;
// arrays below this go the runtime's way, which copies them through its own pinned
// memory (0.79 MB: 51 us, in chunks 56; 1.4 MB: 93 and 89)
constexpr size_t STAGE_MIN = 1 << 20;

}  // namespace

bool pinned_array(const void *p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type == hipMemoryTypeHost || a.type == hipMemoryTypeManaged || a.type == hipMemoryTypeDevice;
}

bool pinned_range(const void *p, size_t bytes) {
    hsa_amd_pointer_info_t info{};
    info.size = sizeof(info);
    if (hsa_amd_pointer_info(p, &info, nullptr, nullptr, nullptr) != HSA_STATUS_SUCCESS) return false;
    if (info.type != HSA_EXT_POINTER_TYPE_HSA || !info.hostBaseAddress ||
        info.agentBaseAddress != info.hostBaseAddress)
        return false;
    const char *base = static_cast<const char *>(info.hostBaseAddress), *q = static_cast<const char *>(p);
    return q >= base && bytes <= info.sizeInBytes && (size_t)(q - base) <= info.sizeInBytes - bytes;
}

bool copy_small_to_host(const std::vector<CopyItem> &items, hipStream_t st) {
    CopyList l{};
    uint64_t bytes = 0;
    for (const CopyItem &c : items) {
        if (l.n == CopyList::MAX || (bytes += c.bytes) > SMALL_MAX) return false;
        // (the kernel writes all of it: a first byte that is pinned is not enough)
        if (!pinned_range(c.dst, c.bytes)) return false;
        if (((uintptr_t)c.dst | (uintptr_t)c.src) % 16) return false;
        l.src[l.n] = c.src;
        l.dst[l.n] = c.dst;
        l.bytes[l.n] = (uint32_t)c.bytes;
        l.block[l.n + 1] = l.block[l.n] + (uint32_t)((c.bytes + CopyList::BLOCK_BYTES - 1) / CopyList::BLOCK_BYTES);
        l.n++;
    }
    if (l.n == 0) return true;
    launch_copy_in(l, nullptr, st);
    HIP_CHECK(hipGetLastError());
    return true;
}

struct HostCopy {
    char *buf = nullptr;
    hipEvent_t ev[SLOTS] = {};
    bool busy[SLOTS] = {};
    int next = 0;

    char *slot(int s) { return buf + (size_t)s * CHUNK; }
    // the slot's last copy is done
    void wait(int s) {
        if (busy[s]) HIP_CHECK(hipEventSynchronize(ev[s]));
        busy[s] = false;
    }
    void mark(int s, hipStream_t st) {
        HIP_CHECK(hipEventRecord(ev[s], st));
        busy[s] = true;
    }
};

void hostcopy_free(HostCopy *h) {
    if (!h) return;
    for (hipEvent_t e : h->ev)
        if (e) (void)hipEventDestroy(e);
    if (h->buf) (void)hipHostFree(h->buf);
    delete h;
}

static HostCopy *hostcopy_get(gis_ctx *ctx) {
    if (!ctx->host_copy) {
        HostCopy *h = new HostCopy();
        ctx->host_copy = h;
        for (hipEvent_t &e : h->ev) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    if (!ctx->host_copy->buf)
        HIP_CHECK(hipHostMalloc((void **)&ctx->host_copy->buf, SLOTS * CHUNK, hipHostMallocDefault));
    return ctx->host_copy;
}

// Chunks of a transfer through the slots in turn: issue(c, slot) puts chunk c's work
// on the stream, and when that is done, finish(c, slot) runs on the host, for a
// longer transfer on threads of its own.
template <typename Issue, typename Finish>
static void pipeline(gis_ctx *ctx, hipStream_t st, uint64_t chunks, Issue issue, Finish finish) {
    std::lock_guard<std::mutex> lock(ctx->host_copy_mu);  // (serving threads copy without the context's lock)
    HostCopy *h = hostcopy_get(ctx);
    const int first = h->next;
    auto slot = [&](uint64_t c) { return (int)((first + c) % SLOTS); };
    std::vector<std::atomic<uint8_t>> state(chunks);  // 1: issued, 2: done
    std::atomic<uint64_t> taken{0};
    std::atomic<int> err{(int)hipSuccess};
    std::atomic<bool> stop{false};
    auto take = [&](uint64_t c) {
        const hipError_t e = hipEventSynchronize(h->ev[slot(c)]);
        if (e == hipSuccess) finish(c, h->slot(slot(c)));
        else err = (int)e;
        h->busy[slot(c)] = false;  // (its next copy waits for state 2)
        state[c].store(2, std::memory_order_release);
    };
    // (a chunk is there within some tens of microseconds, unless the GPU is busy with
    // other work: then the threads leave their cores alone)
    auto wait_for = [&](uint64_t c, uint8_t s) {
        const auto t0 = std::chrono::steady_clock::now();
        bool late = false;
        for (unsigned turn = 1; state[c].load(std::memory_order_acquire) < s && !stop; turn++) {
            if (late) {
                std::this_thread::sleep_for(std::chrono::microseconds(50));
                continue;
            }
            std::this_thread::yield();
            late = turn % 64 == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(500);
        }
        return state[c].load(std::memory_order_acquire) >= s;
    };
    std::vector<std::thread> th;
    struct Join {
        std::vector<std::thread> &th;
        std::atomic<bool> &stop;
        ~Join() {
            stop = true;
            for (std::thread &t : th) t.join();
        }
    };
    {
        Join join{th, stop};
        if (chunks >= THREADS_MIN) {
            try {
                for (int t = 0; t < THREADS; t++)
                    th.emplace_back([&] {
                        (void)hipSetDevice(ctx->device);
                        for (uint64_t c; (c = taken.fetch_add(1)) < chunks && wait_for(c, 1);) take(c);
                    });
            } catch (const std::system_error &) {
                // fewer threads, or none
            }
        }
        const bool inline_ = th.empty();
        for (uint64_t c = 0; c < chunks; c++) {
            if (c < SLOTS) h->wait(slot(c));
            else if (inline_) take(c - SLOTS);
            else (void)wait_for(c - SLOTS, 2);
            if (err != (int)hipSuccess) break;
            issue(c, h->slot(slot(c)));
            HIP_CHECK(hipGetLastError());
            h->mark(slot(c), st);
            state[c].store(1, std::memory_order_release);
        }
        if (err == (int)hipSuccess) {
            if (inline_)
                for (uint64_t c = chunks > SLOTS ? chunks - SLOTS : 0; c < chunks; c++) take(c);
            else
                for (uint64_t c = chunks > SLOTS ? chunks - SLOTS : 0; c < chunks; c++) (void)wait_for(c, 2);
        }
    }
    h->next = slot(chunks);
    if (err != (int)hipSuccess) throw HipError{(hipError_t)err.load(), "copy to the host"};
}

void copy_to_host(gis_ctx *ctx, void *dst, const void *src, size_t n, hipStream_t st) {
    if (n < STAGE_MIN || pinned_array(dst)) {
        if (n) HIP_CHECK(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st));
        return;
    }
    auto bytes = [&](uint64_t c) { return std::min<size_t>(CHUNK, n - c * CHUNK); };
    pipeline(
        ctx, st, (n + CHUNK - 1) / CHUNK,
        [&](uint64_t c, char *p) { launch_copy_out(static_cast<const char *>(src) + c * CHUNK, p, bytes(c), st); },
        [&](uint64_t c, const char *p) { std::memcpy(static_cast<char *>(dst) + c * CHUNK, p, bytes(c)); });
}

void lookup_through_host(gis_ctx *ctx, const uint64_t *keys, uint64_t n, uint64_t *positions, hipStream_t st) {
    constexpr uint64_t KEYS = CHUNK / sizeof(uint64_t);
    const DevIndex ix = dev_index(ctx);
    auto count = [&](uint64_t c) { return std::min(KEYS, n - c * KEYS); };
    pipeline(
        ctx, st, (n + KEYS - 1) / KEYS,
        [&](uint64_t c, char *p) {
            std::memcpy(p, keys + c * KEYS, sizeof(uint64_t) * count(c));
            uint64_t *k = reinterpret_cast<uint64_t *>(p);
            launch_find_flat(ix, k, count(c), k, st);
        },
        [&](uint64_t c, const char *p) { std::memcpy(positions + c * KEYS, p, sizeof(uint64_t) * count(c)); });
}

}  // namespace gis
