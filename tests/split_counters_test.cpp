// The table of csrc/split_counters.h with a runtime that only keeps a record; run by tests/test_native_front_end.py.
#include "split_counters.h"

#include <cstdio>
#include <memory>

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

struct Recorder {
    int device = 0;
    void* captured = (void*)1;  // the stream under capture
    std::vector<std::unique_ptr<uint32_t[]>> memory;
    int current_device() const { return device; }
    bool capturing(void* stream) const { return stream == captured; }
    std::vector<void*> touched;  // the streams that work was put on
    bool no_memory = false, no_clear = false;
    int released = 0;
    uint32_t* allocate(size_t words, void* stream)
    {
        touched.push_back(stream);
        if (no_memory) return nullptr;
        memory.emplace_back(new uint32_t[words]);
        memory.back()[0] = 1;
        return memory.back().get();
    }
    void release(uint32_t*) { ++released; }
    bool clear(uint32_t* p, size_t words, void* stream)
    {
        touched.push_back(stream);
        if (no_clear) return false;
        for (size_t i = 0; i < words; ++i) p[i] = 0;
        return true;
    }
};

static void* stream(long i) { return (void*)(i * 16); }

int main()
{
    fa::CounterTable<Recorder> table;
    Recorder rt;
    // streams of torch's own and the default stream: a region each, the same one call after call
    uint32_t* const a = table.of(rt, 0, stream(1), true);
    uint32_t* const b = table.of(rt, 0, nullptr, false);
    CHECK(a && b && (b - a >= fa::kCountersPerStream || a - b >= fa::kCountersPerStream));
    CHECK(table.of(rt, 0, stream(1), true) == a && table.of(rt, 0, nullptr, false) == b);
    // each cleared on its own stream, once; with nothing to be had the next call tries again
    CHECK(a[0] == 0 && b[0] == 0);
    CHECK((rt.touched == std::vector<void*>{stream(1), stream(1), nullptr, nullptr}));
    rt.no_memory = true;
    CHECK(!table.of(rt, 0, stream(2), true));
    rt.no_memory = false, rt.no_clear = true;
    CHECK(!table.of(rt, 0, stream(2), true) && rt.released == 1);
    rt.no_clear = false;
    CHECK(table.of(rt, 0, stream(2), true) != nullptr);
    // somebody else's stream, a stream under capture
    CHECK(!table.of(rt, 0, stream(7), false));
    rt.captured = stream(1);
    CHECK(!table.of(rt, 0, stream(1), true));
    rt.captured = stream(3);
    const size_t before = rt.touched.size();
    CHECK(!table.of(rt, 0, stream(3), true) && rt.touched.size() == before);
    rt.captured = (void*)1;
    // tensors of another device than the current one: the null stream is not that device's
    rt.device = 1;
    CHECK(!table.of(rt, 0, nullptr, false));
    uint32_t* const c = table.of(rt, 1, nullptr, false);
    CHECK(c && c != b);
    rt.device = 0;
    CHECK(table.of(rt, 0, nullptr, false) == b);
    // no more regions than streams there is room for
    int given = 3;
    for (long i = 3; i < 200; ++i) given += table.of(rt, 0, stream(i), true) != nullptr;
    CHECK(given == fa::kCounterStreams && table.of(rt, 0, stream(1), true) == a);
    return 0;
}
