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
        Device& d = devices_[(size_t)device];
        size_t i = 0;
        while (i < d.streams.size() && d.streams[i] != stream) ++i;
        if (i == d.streams.size()) {
            if (i == (size_t)kCounterStreams) return nullptr;
            if (!d.zeros && !(d.zeros = rt.zeros(device, (size_t)kCountersPerStream * kCounterStreams))) return nullptr;
            d.streams.push_back(stream);
        }
        return d.zeros + i * kCountersPerStream;
    }

private:
    struct Device {
        uint32_t* zeros = nullptr;
        std::vector<void*> streams;
    };
    std::vector<Device> devices_;
};

}  // namespace fa
