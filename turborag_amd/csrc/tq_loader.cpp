// tq_loader.cpp — layer-pipelined load of compressed KV into cache layout.
//
// The reference loads a document layer by layer (tq_backend/cag_store.py:
// 161-288): read the layer's .bin pages, copy them to the GPU (pageable,
// synchronous), dequantize to [N, H, D], then permute to the DynamicCache
// layout [1, H, N, D] with an extra copy.  Here one call enqueues every
// layer: layer l's pages go host -> device on the copy stream while layer
// l-1 is dequantized on the compute stream straight into [1, H, N, D]; the
// compute stream waits for each layer's copy through an event.  With pinned
// host pages (hipHostMalloc / torch pin_memory) the copies run at link rate
// and overlap the dequant.
//
// Layers whose pages follow one another in one pinned host buffer and in one
// device buffer (a store's staging buffers) go as groups: one copy, one event
// and one multi-layer dequant per group.  A copy and its event cost 15-20 us
// beside the bytes, as much as 1 MB of link time (57 GB/s), so small layers
// were bound by their number; the last group's dequant is the one that no copy
// hides, so a group is not the whole document.  Whole calls from Python: 24
// layers of 1.3 MB 1,087-1,112 -> 709-718 us (0.55 ms of link time); 36 of 0.3 MB
// 1,031-1,071 -> 371-380; 36 of 2.2 MB 2,146-2,159 -> 1,605-1,610; 8 of 8.8 MB
// 1,441-1,453 -> 1,367-1,370.
#include <algorithm>
#include <map>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "tq_internal.h"

namespace {

// Per-device events of the loader.  A call holds its device's lock for its
// whole enqueue loop, so two concurrent calls never record and wait on the
// same event in between each other's record and wait (a stream wait takes
// the event's state when it is enqueued, so the events can be re-recorded by
// the next call).  The per-device records never move once created.
struct DeviceEvents {
    std::mutex mu;
    std::vector<hipEvent_t> ev;
};

DeviceEvents& device_events(int dev) {
    static std::mutex mu;
    static std::map<int, std::unique_ptr<DeviceEvents>> all;
    std::lock_guard<std::mutex> lock(mu);
    auto& p = all[dev];
    if (!p) p.reset(new DeviceEvents());
    return *p;
}

void check(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        (void)hipGetLastError();
        throw tq::Error(std::string(what) + ": " + hipGetErrorString(e));
    }
}

// A group's copy: at least this many bytes, unless the layers run out (4 MB
// 805 us for the 24 layers, 10 MB 751, 24 MB 724, all in one 706; 8 layers of
// 9.4 MB 1,644, 1,510, 1,479, 1,480).
constexpr size_t kGroupBytes = size_t(24) << 20;

// The bytes from p to the end of its allocation if p lies in pinned host
// memory (host) or device memory, else 0 (pageable or unknown memory).
size_t bytes_left(const void* p, bool host) {
    hipPointerAttribute_t a{};
    void* start = nullptr;
    size_t size = 0;
    const hipDeviceptr_t d = const_cast<void*>(p);
    const bool ok = hipPointerGetAttributes(&a, p) == hipSuccess &&
                    a.type == (host ? hipMemoryTypeHost : hipMemoryTypeDevice) &&
                    hipPointerGetAttribute(&start, HIP_POINTER_ATTRIBUTE_RANGE_START_ADDR, d) ==
                        hipSuccess &&
                    hipPointerGetAttribute(&size, HIP_POINTER_ATTRIBUTE_RANGE_SIZE, d) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        return 0;
    }
    const size_t at = (size_t)(static_cast<const uint8_t*>(p) - static_cast<uint8_t*>(start));
    return at < size ? size - at : 0;
}

}  // namespace

namespace tq {

void load_layers(Scheme s, const uint8_t* const* host_pools, uint8_t* const* device_pools,
                 size_t pool_bytes, int num_layers, const int32_t* slots, int num_tokens,
                 uint16_t* const* out_key, uint16_t* const* out_value, const PageGeom& g,
                 hipStream_t copy_stream, hipStream_t compute_stream) {
    if (num_layers <= 0) return;
    for (int l = 0; l < num_layers; ++l)
        if (!host_pools[l] || !device_pools[l] || !out_key[l] || !out_value[l])
            throw Error("load_layers: null pool or output pointer for a layer");
    int dev = 0;
    check(hipGetDevice(&dev), "hipGetDevice");
    DeviceEvents& de = device_events(dev);
    std::lock_guard<std::mutex> lock(de.mu);  // held until every layer is enqueued
    std::vector<hipEvent_t>& ev = de.ev;
    while (ev.size() < (size_t)num_layers + 1) {
        hipEvent_t e = nullptr;
        check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreateWithFlags");
        ev.push_back(e);
    }
    const bool two = copy_stream != compute_stream;
    if (two) {
        // Copies must not overwrite pools that earlier compute work still reads.
        check(hipEventRecord(ev[num_layers], compute_stream), "hipEventRecord");
        check(hipStreamWaitEvent(copy_stream, ev[num_layers], 0), "hipStreamWaitEvent");
    }
    // Layers [l, l + n): pages one after another on both sides, inside one
    // allocation each (so that one copy is the n copies), and outputs that meet
    // neither each other nor the pages (a group's layers are dequantized in
    // any order; layers that share a buffer are taken one by one).
    const size_t out_bytes = (size_t)std::max(num_tokens, 0) * g.H * g.D * sizeof(uint16_t);
    const auto meet = [](const void* a, size_t an, const void* b, size_t bn) {
        const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
        return x < y + bn && y < x + an;
    };
    std::vector<std::pair<uintptr_t, uintptr_t>> taken;  // the group's outputs, sorted
    const auto take = [&](const void* p) {
        const uintptr_t x = reinterpret_cast<uintptr_t>(p);
        const std::pair<uintptr_t, uintptr_t> r{x, x + out_bytes};
        const auto at = std::lower_bound(taken.begin(), taken.end(), r);
        if (at != taken.end() && at->first < r.second) return false;
        if (at != taken.begin() && (at - 1)->second > x) return false;
        taken.insert(at, r);
        return true;
    };
    const auto group_at = [&](int l) {
        taken.clear();
        int n = 0;
        while (l + n < num_layers && (n == 0 || n * pool_bytes < kGroupBytes) &&
               host_pools[l + n] == host_pools[l] + n * pool_bytes &&
               device_pools[l + n] == device_pools[l] + n * pool_bytes && take(out_key[l + n]) &&
               take(out_value[l + n]))
            ++n;
        for (const auto& r : taken)
            if (meet(device_pools[l], n * pool_bytes, reinterpret_cast<void*>(r.first), out_bytes))
                return 1;
        return std::max(n, 1);
    };
    size_t host_left = 0, dev_left = 0;  // of the allocations from layer `known` on
    int known = -1;
    for (int l = 0; l < num_layers;) {
        int n = group_at(l);
        if (n > 1) {
            if (known < 0 || host_pools[l] != host_pools[known] + (l - known) * pool_bytes ||
                device_pools[l] != device_pools[known] + (l - known) * pool_bytes) {
                host_left = bytes_left(host_pools[l], true);
                dev_left = bytes_left(device_pools[l], false);
                known = l;
            }
            const size_t end = (size_t)(l - known + n) * pool_bytes;
            if (end > host_left || end > dev_left) n = 1;
        }
        check(hipMemcpyAsync(device_pools[l], host_pools[l], n * pool_bytes, hipMemcpyHostToDevice,
                             copy_stream),
              "hipMemcpyAsync");
        if (two) {
            check(hipEventRecord(ev[l], copy_stream), "hipEventRecord");
            check(hipStreamWaitEvent(compute_stream, ev[l], 0), "hipStreamWaitEvent");
        }
        launch_dequant_layers(s, device_pools + l, slots, out_key + l, out_value + l, g, num_tokens,
                              n, compute_stream, /*head_major=*/true);
        l += n;
    }
}

}  // namespace tq
