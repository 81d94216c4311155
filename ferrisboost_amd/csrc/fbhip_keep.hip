// Memory and streams kept between jobs.
//
// A training job makes some 90 device allocations, 10 page-locked ones and 4
// streams, and gives them all back when it ends. hipMalloc and hipFree wait for
// the driver, which clears memory before it hands it out again: most take 10 to
// 100 us, but once a process has turned over about 70 GB the clearing falls behind
// and single calls take 20 to 970 ms (400k x 2000, 40 rounds: 265 ms for six jobs,
// then 443 and 1085; 2M x 100: 157, then 250 to 2030). A stream costs 0.5 ms to
// make and 0.4 to destroy. So what a job gives back is kept for the next one: those
// jobs now take 256 and 132 ms each time, 10.5M x 28, 100 rounds 283 -> 266,
// 100k x 28, 100 rounds 50 -> 42 and 5k x 20, 50 rounds 19 -> 17.
//
// Blocks serve requests of their own size alone, so nobody holds more memory than
// was asked for. A device keeps at most a sixteenth of its memory, the oldest
// blocks beyond that go; a failed allocation, an object with a memory budget and
// fbh_release_cached give everything back, parked models (fbh_shap_model_park) first. Who gives a block or a stream back has
// waited for all work on it, so any thread and stream can take it next. Contents
// are those of the last use, as of any block that hipMalloc cuts from a page in use.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <iterator>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/fbhip.h"
#include "fbhip_internal.h"

namespace fbh {

namespace {

constexpr int MAX_KEEP_DEVICES = 64;
constexpr uint64_t DEVICE_SHARE = 16;              // of a device's memory, kept at most
constexpr uint64_t HOST_MOST = 64ull << 20;        // page-locked bytes kept
constexpr size_t STREAMS_MOST = 8;                 // streams kept of a device
constexpr size_t BLOCKS_MOST = 1024;               // blocks kept of a device

struct Block {
    void *p;
    uint64_t bytes;
    KeepKind kind;
    int device;
};

struct Kept {
    std::mutex mu;
    std::unordered_map<void *, Block> out;  // blocks in use
    std::vector<Block> in[MAX_KEEP_DEVICES];  // kept, oldest first
    uint64_t bytes[MAX_KEEP_DEVICES] = {}, host_bytes = 0;
    uint64_t most[MAX_KEEP_DEVICES] = {};  // 0: not asked yet
    std::vector<hipStream_t> streams[MAX_KEEP_DEVICES];
};

// Never destroyed: the runtime may be gone when a process' static objects are.
Kept &kept() {
    static Kept *k = new Kept;
    return *k;
}

void give_back(const Block &b) {
    if (b.kind == KeepKind::device) (void)hipFree(b.p);
    else (void)hipHostFree(b.p);
}

uint64_t &bytes_of(Kept &k, const Block &b) {
    return b.kind == KeepKind::device ? k.bytes[b.device] : k.host_bytes;
}

hipError_t make(KeepKind kind, void **p, uint64_t bytes) {
    switch (kind) {
        case KeepKind::device: return hipMalloc(p, bytes);
        case KeepKind::host: return hipHostMalloc(p, bytes, hipHostMallocDefault);
        default: return hipHostMalloc(p, bytes, hipHostMallocCoherent);
    }
}

}  // namespace

hipError_t keep_alloc(KeepKind kind, void **p, uint64_t bytes) {
    *p = nullptr;
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return e;
    bytes = (bytes + 255) & ~uint64_t(255);
    if (dev >= MAX_KEEP_DEVICES) return make(kind, p, bytes);
    Kept &k = kept();
    {
        std::lock_guard<std::mutex> g(k.mu);
        std::vector<Block> &in = k.in[dev];
        for (size_t i = in.size(); i-- > 0;)
            if (in[i].bytes == bytes && in[i].kind == kind) {
                k.out.emplace(in[i].p, in[i]);  // (throws before the block leaves the list)
                *p = in[i].p;
                bytes_of(k, in[i]) -= bytes;
                in.erase(in.begin() + (ptrdiff_t)i);
                return hipSuccess;
            }
    }
    hipError_t e = make(kind, p, bytes);
    if (e != hipSuccess && keep_release(dev)) {
        (void)hipGetLastError();
        e = make(kind, p, bytes);
    }
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> g(k.mu);
    try {
        k.out.emplace(*p, Block{*p, bytes, kind, dev});
    } catch (...) {
        give_back({*p, bytes, kind, dev});
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    return hipSuccess;
}

void keep_free(KeepKind kind, void *p, bool keep) noexcept {
    if (!p) return;
    Kept &k = kept();
    Block b{p, 0, kind, 0};
    uint64_t total = 0;
    {
        std::lock_guard<std::mutex> g(k.mu);
        const auto it = k.out.find(p);
        if (it == k.out.end()) keep = false;
        else {
            b = it->second;
            k.out.erase(it);
            total = k.most[b.device];
        }
    }
    if (keep && !total) {
        size_t free_b = 0, total_b = 0;
        int dev = -1;
        // (the caller has made the block's device current)
        if (hipGetDevice(&dev) != hipSuccess || dev != b.device ||
            hipMemGetInfo(&free_b, &total_b) != hipSuccess)
            keep = false;
        else total = total_b / DEVICE_SHARE;
    }
    const uint64_t most = b.kind == KeepKind::device ? total : HOST_MOST;
    if (!keep || b.bytes > most) {
        give_back(b);
        return;
    }
    std::vector<Block> old;
    {
        std::lock_guard<std::mutex> g(k.mu);
        k.most[b.device] = total;
        std::vector<Block> &in = k.in[b.device];
        try {
            old.reserve(in.size() + 1);
            in.push_back(b);
            bytes_of(k, b) += b.bytes;
        } catch (...) {
            old.clear();
            keep = false;
        }
        for (size_t i = 0; keep && i < in.size();) {
            const bool alike = (in[i].kind == KeepKind::device) == (b.kind == KeepKind::device);
            if (in.size() <= BLOCKS_MOST && !(alike && bytes_of(k, b) > most)) {
                i++;
                continue;
            }
            bytes_of(k, in[i]) -= in[i].bytes;
            old.push_back(in[i]);
            in.erase(in.begin() + (ptrdiff_t)i);
        }
    }
    if (!keep) give_back(b);
    for (const Block &o : old) give_back(o);
}

bool keep_release(int device) noexcept {
    const bool models = drop_parked(device);  // (their memory is kept, and goes below)
    if (device < 0 || device >= MAX_KEEP_DEVICES) return models;
    Kept &k = kept();
    std::vector<Block> in;
    std::vector<hipStream_t> streams;
    {
        std::lock_guard<std::mutex> g(k.mu);
        in.swap(k.in[device]);
        streams.swap(k.streams[device]);
        for (const Block &b : in) bytes_of(k, b) -= b.bytes;
    }
    for (const Block &b : in) give_back(b);
    for (hipStream_t s : streams) (void)hipStreamDestroy(s);
    return models || !in.empty();
}

uint64_t keep_bytes(int device) noexcept {
    const uint64_t models = parked_bytes(device);
    if (device < 0 || device >= MAX_KEEP_DEVICES) return models;
    Kept &k = kept();
    std::lock_guard<std::mutex> g(k.mu);
    return models + k.bytes[device];
}

hipError_t keep_stream(hipStream_t *s) {
    *s = nullptr;
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return e;
    if (dev < MAX_KEEP_DEVICES) {
        Kept &k = kept();
        std::lock_guard<std::mutex> g(k.mu);
        if (!k.streams[dev].empty()) {
            *s = k.streams[dev].back();
            k.streams[dev].pop_back();
            return hipSuccess;
        }
    }
    return hipStreamCreateWithFlags(s, hipStreamNonBlocking);
}

hipError_t keep_stream_back(int device, hipStream_t s, bool idle) noexcept {
    if (!s) return hipSuccess;
    // Waits for it (0.4 us when there is nothing to wait for); a stream that reports an
    // error is not handed on.
    const hipError_t e = idle ? hipSuccess : hipStreamSynchronize(s);
    if (e == hipSuccess && device >= 0 && device < MAX_KEEP_DEVICES) {
        Kept &k = kept();
        std::lock_guard<std::mutex> g(k.mu);
        try {
            if (k.streams[device].size() < STREAMS_MOST) {
                k.streams[device].push_back(s);
                return e;
            }
        } catch (...) {
        }
    }
    (void)hipStreamDestroy(s);
    return e;
}

}  // namespace fbh

extern "C" int fbh_release_cached(int device) {
    (void)fbh::keep_release(device);
    return FBH_OK;
}
