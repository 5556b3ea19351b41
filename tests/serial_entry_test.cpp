// A userdriver serialises its own entry points (include/eden_ud.h), on a CPU: the device calls behind them are stood in for,
// and while one thread records a list's graph another one makes each of the other calls.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <thread>
#include <utility>
#include <vector>

#include "eden_hip.h"
#include "eden_ud.h"

namespace {
std::atomic<bool> recording{false};
std::atomic<int> intruders{0};          // device calls of another thread that reached the stream during the recording
std::function<void()> while_recording;  // called from inside a recording
thread_local bool recorder = false;
std::vector<std::function<void()>> recorded;

void arrive() {
    if (recording && !recorder) ++intruders;
}
int enqueue(std::function<void()> work) {
    arrive();
    if (recording)
        recorded.push_back(work);
    else
        work();
    return EH_OK;
}
struct Slot {
    size_t bytes;
    void *memory;
};
}  // namespace

struct eh_pool {
    std::vector<Slot> slots;
};

extern "C" {
int eh_init(int) { return EH_OK; }
const char *eh_last_error(void) { return ""; }
int eh_stream_create(void **s) { return *s = std::malloc(1), EH_OK; }
int eh_stream_destroy(void *s) { return std::free(s), EH_OK; }
int eh_stream_sync(void *) { return arrive(), EH_OK; }
int eh_stream_idle(void *, int32_t *idle) { return *idle = 1, EH_OK; }
int eh_event_create_untimed(void **e) { return *e = std::malloc(1), EH_OK; }
int eh_event_destroy(void *e) { return std::free(e), EH_OK; }
int eh_event_record(void *, void *) { return EH_OK; }
int eh_stream_wait_event(void *, void *) { return EH_OK; }
int eh_host_alloc(void **p, size_t bytes) { return *p = std::malloc(bytes), EH_OK; }
int eh_host_free(void *p) { return std::free(p), EH_OK; }
int eh_malloc(void **p, size_t bytes) { return *p = std::calloc(1, bytes), EH_OK; }
int eh_free(void *p) { return std::free(p), EH_OK; }
int eh_copy_pinned(void *dst, const void *src, size_t bytes, void *) {
    return enqueue([=] { std::memcpy(dst, src, bytes); });
}
int eh_h2d(void *dst, const void *src, size_t bytes, void *s) { return eh_copy_pinned(dst, src, bytes, s); }
int eh_d2h(void *dst, const void *src, size_t bytes, void *s) { return eh_copy_pinned(dst, src, bytes, s); }
int eh_add_u8(const void *a, const void *b, void *out, int64_t count, const eh_add_requant *, void *) {
    if (recording && recorder && while_recording) std::exchange(while_recording, nullptr)();
    return enqueue([=] {
        for (int64_t i = 0; i < count; ++i) static_cast<uint8_t *>(out)[i] = (uint8_t)(static_cast<const uint8_t *>(a)[i] + static_cast<const uint8_t *>(b)[i]);
    });
}
int eh_graph_begin(void *) {
    recorded.clear();
    recorder = true;
    recording = true;
    return EH_OK;
}
int eh_graph_end(void *, void **graph) {
    recording = false;
    recorder = false;
    *graph = new std::vector<std::function<void()>>(recorded);
    return EH_OK;
}
int eh_graph_launch(void *graph, void *) {
    for (auto &work : *static_cast<std::vector<std::function<void()>> *>(graph)) work();
    return EH_OK;
}
int eh_graph_destroy(void *graph) { return delete static_cast<std::vector<std::function<void()>> *>(graph), EH_OK; }
int eh_pool_create(eh_pool **pool) { return *pool = new eh_pool, EH_OK; }
int eh_pool_request(eh_pool *pool, int, size_t bytes, int32_t *slot) {
    *slot = (int32_t)pool->slots.size();
    pool->slots.push_back({bytes, nullptr});
    return EH_OK;
}
int eh_pool_reset_inter(eh_pool *, int32_t) { return EH_OK; }
int eh_pool_reset_intra(eh_pool *) { return EH_OK; }
int eh_pool_assign(eh_pool *pool, size_t *bytes) {
    *bytes = 0;
    for (auto &s : pool->slots)
        if (!s.memory) s.memory = std::calloc(1, s.bytes ? s.bytes : 1), *bytes += s.bytes;
    return EH_OK;
}
int eh_pool_slot(const eh_pool *pool, int32_t slot, void **p, size_t *bytes) {
    if (p) *p = pool->slots[(size_t)slot].memory;
    if (bytes) *bytes = pool->slots[(size_t)slot].bytes;
    return EH_OK;
}
int eh_pool_release(eh_pool *pool, int32_t slot) {
    std::free(pool->slots[(size_t)slot].memory);
    pool->slots[(size_t)slot].memory = nullptr;
    return EH_OK;
}
int eh_pool_destroy(eh_pool *pool) {
    for (auto &s : pool->slots) std::free(s.memory);
    return delete pool, EH_OK;
}
}

static int failures = 0;
static void expect(bool ok, const char *what) {
    if (!ok) std::printf("FAILED: %s\n", what);
    failures += !ok;
}

int main() {
    eud_driver *driver = nullptr;
    expect(eud_initialize(&driver, 0) == 0, "initialize");
    const uint32_t shape[4] = {1, 1, 1, 64};
    auto open = [&](uint64_t id) {
        eud_oplist *list = nullptr;
        expect(eud_oplist_create(&list, id, EUD_MODEL_ANDROID_NN) == 0, "create");
        int32_t t[3];
        for (int32_t i = 0; i < 3; ++i) t[i] = eud_oplist_feature_map(list, i, shape, 4, EUD_TENSOR_UINT8, 0.5f, 0);
        const eud_options options{};
        expect(eud_oplist_operator(list, "ADD", EUD_OP_ADD, t, 2, t + 2, 1, &options) == 0, "operator");
        expect(eud_open_subgraph(driver, list, 1) == 0, "open");
        eud_oplist_destroy(list);
    };
    const struct {
        const char *name;
        std::function<int()> call;
    } calls[] = {
        {"eud_write_input", [&] { uint8_t in[64] = {9}; return eud_write_input(driver, 1, 0, in, 64); }},
        {"eud_read_output", [&] { uint8_t out[64]; return eud_read_output(driver, 1, 0, out, 64); }},
        {"eud_synchronize", [&] { return eud_synchronize(driver); }},
        {"eud_execute_operators", [&] { return eud_execute_operators(driver, 1, 1); }},
    };
    open(1);
    uint64_t id = 2;
    for (const auto &other : calls) {
        open(id);
        std::vector<uint8_t> a(64, 1), b(64, 2), c(64, 0);
        const int32_t indices[3] = {0, 1, 2};
        void *addresses[3] = {a.data(), b.data(), c.data()};
        const size_t sizes[3] = {64, 64, 64};
        std::thread beside;
        intruders = 0;
        int result = -1;
        while_recording = [&] {
            beside = std::thread([&] { result = other.call(); });
            std::this_thread::sleep_for(std::chrono::milliseconds(100));  // (long enough for the call to come through if nothing holds it)
        };
        for (int rep = 0; rep < 4; ++rep) {
            std::fill(c.begin(), c.end(), 0);
            expect(eud_execute_subgraph(driver, id, indices, addresses, sizes, 3) == 0, other.name);
            expect(c == std::vector<uint8_t>(64, 3), other.name);
        }
        expect(beside.joinable(), "the list was recorded");
        if (beside.joinable()) beside.join();
        expect(result == 0, other.name);
        if (intruders) std::printf("FAILED: %s reached the stream while another thread recorded a graph\n", other.name);
        failures += intruders != 0;
        expect(eud_close_subgraph(driver, id) == 0, "close");
        ++id;
    }
    eud_deinitialize(driver);
    if (!failures) std::printf("ok\n");
    return failures != 0;
}
