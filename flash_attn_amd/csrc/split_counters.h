// Arrival counters (flash_params::split_counters) of the calls that the Python front end makes, one region of kCountersPerStream
// zeros for each of up to kCounterStreams streams of a device.
// Runtime is what the table asks of the GPU's runtime (py_binding.cpp; tests/split_counters_test.cpp has one without a GPU).
#pragma once
#include <cstddef>
#include <cstdint>
#include <vector>

namespace fa {

constexpr int kCountersPerStream = 4096, kCounterStreams = 64;

// Only the default stream and torch's own pooled streams get a region: those exist until the process ends, so calls that
// share one are ordered for good.  Other streams, calls under graph capture (a graph may be replayed beside other work) and
// whoever comes too late merge in a launch of their own: nullptr.
template <class Runtime>
class CounterTable {
public:
    uint32_t* of(Runtime& rt, int device, void* stream, bool pooled)
    {
        if (stream != nullptr && !pooled) return nullptr;
        // A call runs on the current device, and the null stream is that device's: with tensors of another device two null
        // streams, which nothing orders, would be one entry of the tensors' device.
        if (rt.current_device() != device) return nullptr;
        if (rt.capturing(stream)) return nullptr;
        if ((size_t)device >= devices_.size()) devices_.resize((size_t)device + 1);
        std::vector<Region>& regions = devices_[(size_t)device];
        for (const Region& r : regions)
            if (r.stream == stream) return r.counters;
        if (regions.size() == (size_t)kCounterStreams) return nullptr;
        // Allocated and cleared on the stream itself, in front of the launches that count in it: no other stream is touched, none
        // waited for (the current one may be another, and under capture).
        uint32_t* const fresh = rt.allocate(kCountersPerStream, stream);
        if (fresh == nullptr) return nullptr;
        if (!rt.clear(fresh, kCountersPerStream, stream)) {
            rt.release(fresh);
            return nullptr;
        }
        regions.push_back({stream, fresh});
        return fresh;
    }

private:
    struct Region {
        void* stream;
        uint32_t* counters;
    };
    std::vector<std::vector<Region>> devices_;
};

}  // namespace fa
