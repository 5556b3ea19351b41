// The runtime's pinned staging area (host/HipRuntime.hpp) on a CPU: the device calls it makes are stood in for by streams
// that run what they were given only when somebody waits for them, the latest a real stream may run it.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <vector>

#include "HipRuntime.hpp"

namespace {
struct Event {
    std::shared_ptr<bool> done;
    void *stream = nullptr;
};
struct Stream {
    std::vector<std::function<void()>> queue;
    void drain() {
        while (!queue.empty()) {
            auto front = queue.front();
            queue.erase(queue.begin());
            front();
        }
    }
};
Stream &as_stream(void *s) { return *static_cast<Stream *>(s); }
}  // namespace

extern "C" {
int eh_init(int) { return EH_OK; }
const char *eh_last_error(void) { return ""; }
int eh_stream_create(void **s) { return *s = new Stream, EH_OK; }
int eh_stream_destroy(void *s) { return delete static_cast<Stream *>(s), EH_OK; }
int eh_stream_sync(void *s) { return as_stream(s).drain(), EH_OK; }
int eh_event_create_untimed(void **e) { return *e = new Event, EH_OK; }
int eh_event_destroy(void *e) { return delete static_cast<Event *>(e), EH_OK; }
int eh_event_record(void *e, void *s) {
    auto done = std::make_shared<bool>(false);
    static_cast<Event *>(e)->done = done;
    static_cast<Event *>(e)->stream = s;
    as_stream(s).queue.push_back([done] { *done = true; });
    return EH_OK;
}
int eh_stream_wait_event(void *s, void *e) {
    const Event at = *static_cast<Event *>(e);
    as_stream(s).queue.push_back([at] {
        if (!*at.done) as_stream(at.stream).drain();
    });
    return EH_OK;
}
int eh_host_alloc(void **p, size_t bytes) { return *p = std::malloc(bytes), EH_OK; }
int eh_host_free(void *p) { return std::free(p), EH_OK; }
int eh_malloc(void **p, size_t bytes) { return *p = std::calloc(1, bytes), EH_OK; }
int eh_free(void *p) { return std::free(p), EH_OK; }
int eh_copy_pinned(void *dst, const void *src, size_t bytes, void *s) {
    as_stream(s).queue.push_back([=] { std::memcpy(dst, src, bytes); });
    return EH_OK;
}
int eh_h2d(void *dst, const void *src, size_t bytes, void *s) { return eh_copy_pinned(dst, src, bytes, s); }
int eh_d2h(void *dst, const void *src, size_t bytes, void *s) { return eh_copy_pinned(dst, src, bytes, s); }
int eh_pool_destroy(eh_pool *) { return EH_OK; }
}

using enn::ud::hip::HipRuntime;

static int failures = 0;
static void expect(bool ok, const char *what) {
    if (!ok) std::printf("FAILED: %s\n", what);
    failures += !ok;
}
static bool all(const std::vector<char> &v, char value) {
    for (char c : v)
        if (c != value) return false;
    return true;
}

// A lane's input is on its way (not joined to the main stream yet) while another thread transfers and waits.
static void lane_write_beside(const std::function<void(HipRuntime &)> &other, const char *what) {
    HipRuntime rt;
    rt.initialize(0);
    rt.initializeQueue();
    const size_t bytes = 1 << 20;
    const std::vector<char> a(bytes, 'a'), b(bytes, 'b');
    std::vector<char> lane_input(bytes, 0), main_input(bytes, 0);
    void *lane = rt.laneStream(0);
    expect(rt.writeBufferOn(lane_input.data(), a.data(), bytes, lane) == Status::SUCCESS, what);
    other(rt);
    expect(rt.writeBuffer(main_input.data(), b.data(), 1, (uint32_t)bytes, false) == Status::SUCCESS, what);
    eh_event_record(rt.event(1), lane);
    eh_stream_wait_event(rt.mainStream(), rt.event(1));
    rt.lanesJoined();
    expect(rt.synchronize() == Status::SUCCESS, what);
    expect(all(lane_input, 'a') && all(main_input, 'b'), what);
}

int main() {
    lane_write_beside([](HipRuntime &) {}, "nothing else");
    lane_write_beside([](HipRuntime &rt) { rt.synchronize(); }, "a synchronization before the join");
    lane_write_beside(
        [](HipRuntime &rt) {
            std::vector<char> x(4096, 'x'), dev(4096, 0);
            rt.writeBuffer(dev.data(), x.data(), 1, 4096, true);
            expect(all(dev, 'x'), "the blocking write itself");
        },
        "a blocking write before the join");
    lane_write_beside(
        [](HipRuntime &rt) {
            std::vector<char> x(4096, 'x'), host(4096, 0);
            rt.readBuffer(host.data(), x.data(), 1, 4096, true);
            expect(all(host, 'x'), "the blocking read itself");
        },
        "a blocking read before the join");
    // more than the area holds, in two lanes and on the main stream at once
    {
        HipRuntime rt;
        rt.initialize(0);
        rt.initializeQueue();
        const size_t bytes = (size_t)7 << 20;
        const std::vector<char> a(bytes, 'a'), b(bytes, 'b'), c(bytes, 'c');
        std::vector<char> da(bytes, 0), db(bytes, 0), dc(bytes, 0);
        rt.writeBufferOn(da.data(), a.data(), bytes, rt.laneStream(0));
        rt.writeBufferOn(db.data(), b.data(), bytes, rt.laneStream(1));
        rt.writeBufferOn(dc.data(), c.data(), bytes, rt.mainStream());
        for (size_t lane = 0; lane < 2; ++lane) {
            eh_event_record(rt.event(lane), rt.laneStream(lane));
            eh_stream_wait_event(rt.mainStream(), rt.event(lane));
        }
        rt.lanesJoined();
        rt.synchronize();
        expect(all(da, 'a') && all(db, 'b') && all(dc, 'c'), "writes beyond the area's size");
    }
    // the runtime goes while a lane's copy is queued: its memory must still be there when the copy runs
    {
        const size_t bytes = 4096;
        const std::vector<char> a(bytes, 'a');
        std::vector<char> da(bytes, 0);
        {
            HipRuntime rt;
            rt.initialize(0);
            rt.initializeQueue();
            rt.writeBufferOn(da.data(), a.data(), bytes, rt.laneStream(0));
        }
        expect(all(da, 'a'), "a copy queued when the runtime goes");
    }
    if (!failures) std::printf("ok\n");
    return failures != 0;
}
