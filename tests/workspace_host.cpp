// Host model of the HIP calls that qengine_amd/csrc/workspace.cpp makes, and the scenarios of test_workspace.py on it:
// linked with workspace.cpp by g++, no GPU and no HIP runtime. "Device memory" is malloc; a scenario sets what a stream's
// capture status is and which calls fail.
#include <atomic>
#include <chrono>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../qengine_amd/csrc/qe_api.hpp"

#define EXPECT(c)                                                    \
    do {                                                             \
        if (!(c)) {                                                  \
            printf("FAILED %s:%d %s\n", __FILE__, __LINE__, #c);     \
            exit(1);                                                 \
        }                                                            \
    } while (0)

namespace {
struct Graph {
    int refs = 1;  // the graph and its executables
    std::vector<std::pair<hipHostFn_t, void*>> held;
};
struct Capture {
    unsigned long long id;
    Graph* graph;
};
std::mutex g_model;
std::map<hipStream_t, Capture> g_captures;  // streams being captured
unsigned long long g_next_id = 0;
size_t g_allocs = 0, g_tries = 0, g_held = 0;  // allocations, attempts, bytes held
std::map<void*, size_t> g_sizes;
std::atomic<bool> g_oom{false};
std::map<hipStream_t, int> g_synced;  // synchronizations by stream
thread_local hipStreamCaptureMode t_mode = hipStreamCaptureModeGlobal;

Graph* begin_capture(hipStream_t st) {
    Graph* g = new Graph;
    g_captures[st] = Capture{++g_next_id, g};
    return g;
}
void end_capture(hipStream_t st) { g_captures.erase(st); }
void unref(Graph* g) {  // the graph or an executable of it is destroyed
    if (--g->refs) return;
    for (auto& h : g->held) h.first(h.second);
    delete g;
}
}  // namespace

// ---- the HIP calls ----
extern "C" {
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "model"; }
hipError_t hipStreamGetCaptureInfo_v2(hipStream_t st, hipStreamCaptureStatus* s, unsigned long long* id, hipGraph_t* g,
                                      const hipGraphNode_t**, size_t*) {
    std::lock_guard<std::mutex> lk(g_model);
    auto it = g_captures.find(st);
    *s = it == g_captures.end() ? hipStreamCaptureStatusNone : hipStreamCaptureStatusActive;
    if (it != g_captures.end()) {
        *id = it->second.id;
        *g = reinterpret_cast<hipGraph_t>(it->second.graph);
    }
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    std::swap(*m, t_mode);
    return hipSuccess;
}
hipError_t hipUserObjectCreate(hipUserObject_t* o, void* p, hipHostFn_t f, unsigned, unsigned) {
    *o = reinterpret_cast<hipUserObject_t>(new std::pair<hipHostFn_t, void*>(f, p));
    return hipSuccess;
}
hipError_t hipGraphRetainUserObject(hipGraph_t g, hipUserObject_t o, unsigned, unsigned) {
    auto* h = reinterpret_cast<std::pair<hipHostFn_t, void*>*>(o);
    reinterpret_cast<Graph*>(g)->held.push_back(*h);
    delete h;
    return hipSuccess;
}
// memory calls fail in a thread of the global mode while any stream is being captured, as HIP's do
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> lk(g_model);
    if (t_mode == hipStreamCaptureModeGlobal && !g_captures.empty()) return hipErrorStreamCaptureUnsupported;
    g_tries++;
    if (g_oom) return hipErrorOutOfMemory;
    g_allocs++;
    g_held += n;
    *p = malloc(n);
    g_sizes[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lk(g_model);
    if (t_mode == hipStreamCaptureModeGlobal && !g_captures.empty()) return hipErrorStreamCaptureUnsupported;
    g_held -= g_sizes.at(p);
    g_sizes.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(8);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
    memset(p, v, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
    std::lock_guard<std::mutex> lk(g_model);
    g_synced[st]++;
    return hipSuccess;
}
}
int qe_num_cus() { return 4; }
[[noreturn]] void qe_fatal_check() {
    printf("FATAL\n");
    exit(3);
}
[[noreturn]] void qe_fatal_hip(hipError_t e, const char* what, const char*, int) {
    printf("FATAL HIP %d %s\n", (int)e, what);
    exit(3);
}

static hipStream_t stream(long i) { return reinterpret_cast<hipStream_t>(i * 16); }

// two host threads on one stream: what one call writes into the buffer is still there when its last launch reads it
static void threads_on_one_stream() {
    std::atomic<int> bad{0};
    auto call = [&](int id) {
        for (int i = 0; i < 200; i++) {
            WsHold hold(stream(1));
            int* p = static_cast<int*>(hold.get(kWsSkinny, 64));
            *const_cast<volatile int*>(p) = id;  // the first launch
            std::this_thread::sleep_for(std::chrono::microseconds(20));
            if (*const_cast<volatile int*>(p) != id) bad++;  // the launch that reads it
        }
    };
    std::thread a(call, 1), b(call, 2);
    a.join();
    b.join();
    EXPECT(bad == 0);
}

// a call on another stream does not wait for the hold
static void another_stream_runs() {
    WsHold hold(stream(1));
    void* p = hold.get(kWsSplit, 100);
    std::atomic<bool> done{false};
    std::thread t([&] {
        WsHold h2(stream(2));
        EXPECT(h2.get(kWsSplit, 100) != p);
        done = true;
    });
    t.join();
    EXPECT(done);
    EXPECT(ws_count(kWsSplit) == 2);
}

// every kind under capture: not the stream's buffer, the same one again in that capture, another for another capture and
// another stream; the kinds that need sizing get none before
static void captures_have_their_own() {
    for (int kind = 0; kind < kNumWs; kind++) {
        hipStream_t st = stream(10 + kind), other = stream(100 + kind);
        const bool sizing = kind == kWsSplit || kind == kWsI8 || kind == kWsH;
        Graph* g0 = begin_capture(st);
        EXPECT((WsHold(st).get(kind, 1 << 20) == nullptr) == sizing);
        end_capture(st);
        unref(g0);
        void* own = WsHold(st).get(kind, 1 << 20);
        EXPECT(own && WsHold(other).get(kind, 1 << 20));
        Graph* g1 = begin_capture(st);
        void* a = WsHold(st).get(kind, 1 << 20);
        EXPECT(a && a != own && WsHold(st).get(kind, 1000) == a);
        EXPECT((WsHold(st).get(kind, 64 << 20) == nullptr) == sizing);
        end_capture(st);
        EXPECT(WsHold(st).get(kind, 1 << 20) == own);
        Graph* g2 = begin_capture(st);
        Graph* g3 = begin_capture(other);
        void *b = WsHold(st).get(kind, 1 << 20), *c = WsHold(other).get(kind, 1 << 20);
        EXPECT(b && c && b != c && b != a && c != a && b != own);
        end_capture(st);
        end_capture(other);
        unref(g1), unref(g2), unref(g3);
    }
}

// a graph's buffer serves no other capture while the graph or an executable of it lives, and the next one after that
static void graphs_give_back() {
    hipStream_t st = stream(1);
    const int before = ws_count(kWsDec);
    Graph* g1 = begin_capture(st);
    void* a = WsHold(st).get(kWsDec, 1 << 20);
    end_capture(st);
    g1->refs++;  // instantiated
    unref(g1);   // the graph is destroyed, the executable lives
    Graph* g2 = begin_capture(st);
    void* b = WsHold(st).get(kWsDec, 1 << 20);
    end_capture(st);
    EXPECT(a != b && ws_count(kWsDec) == before + 2);
    unref(g1);
    EXPECT(ws_count(kWsDec) == before + 1);
    const size_t allocs = g_allocs;
    for (int i = 0; i < 5; i++) {
        Graph* g = begin_capture(st);
        EXPECT(WsHold(st).get(kWsDec, 1 << 20) == a);
        end_capture(st);
        unref(g);
    }
    EXPECT(g_allocs == allocs);
    unref(g2);
    EXPECT(ws_count(kWsDec) == before);
}

// a stream's first call while another thread captures on another stream in the global mode
static void allocate_beside_a_capture() {
    Graph* g = begin_capture(stream(1));
    std::thread([] {
        for (int kind = 0; kind < kNumWs; kind++) {
            EXPECT(WsHold(stream(2)).get(kind, 1 << 20) != nullptr);
            EXPECT(WsHold(nullptr).get(kind, 1 << 20) != nullptr);
        }
        EXPECT(t_mode == hipStreamCaptureModeGlobal);
    }).join();
    end_capture(stream(1));
    unref(g);
}

// no memory under capture: no buffer, and the capture goes on
static void capture_without_memory() {
    hipStream_t st = stream(1);
    Graph* g = begin_capture(st);
    g_oom = true;
    EXPECT(WsHold(st).get(kWsSkinny, 1 << 20) == nullptr);
    g_oom = false;
    EXPECT(WsHold(st).get(kWsSkinny, 1 << 20) != nullptr);
    end_capture(st);
    unref(g);
}

static void* get(hipStream_t st, int kind, size_t bytes) { return WsHold(st).get(kind, bytes); }
static size_t sized(hipStream_t st, int kind) { return WsHold(st).sized(kind); }

// a growing call gives the outgrown buffer back once the stream's work on it is done
static void growth_frees() {
    hipStream_t st = stream(1);
    Graph* g = begin_capture(stream(2));  // (freeing beside a capture, too)
    for (int kind = 0; kind < kNumWs; kind++)
        for (size_t mb = 1; mb <= 40; mb++) {
            const size_t held = g_held, own = sized(st, kind);
            const int synced = g_synced[st];
            EXPECT(get(st, kind, mb << 20) && sized(st, kind) == mb << 20);
            EXPECT(g_held == held - own + (mb << 20) && g_synced[st] == synced + (mb > 1));
            EXPECT(get(st, kind, 1 << 20) && g_held == held - own + (mb << 20));
        }
    end_capture(stream(2));
    unref(g);
}

// no memory: the calls that can run without a buffer are told so and do not ask the device each time; they get one later
static void without_memory() {
    for (int kind : {kWsSplit, kWsDec, kWsSkinny}) {
        hipStream_t st = stream(1);
        g_oom = true;
        const size_t tries = g_tries;
        for (int i = 0; i < 1000; i++) EXPECT(get(st, kind, 2 << 20) == nullptr);
        EXPECT(g_tries - tries >= 2 && g_tries - tries <= 10);
        EXPECT(get(st, kind, 1 << 20) == nullptr);
        EXPECT(g_tries - tries <= 11);  // a smaller size is asked for
        g_oom = false;
        int i = 0;
        while (get(st, kind, 2 << 20) == nullptr) EXPECT(++i < 1000);
        EXPECT(get(st, kind, 1 << 20) != nullptr);
        g_oom = true;
        EXPECT(get(st, kind, 3 << 20) == nullptr);
        g_oom = false;
        ws_reserve(kind, 3 << 20, st);  // a reserve asks at once
        g_oom = true;  // growing fails: the smaller buffer stays
        EXPECT(get(st, kind, 4 << 20) == nullptr && get(st, kind, 3 << 20) != nullptr);
        g_oom = false;
    }
}

// what a reserve that cannot be met reports
static void reserve_in_capture() {
    ws_reserve(kWsSplit, 1 << 20, stream(1));
    begin_capture(stream(1));
    ws_reserve(kWsSplit, 1 << 20, stream(1));
    ws_reserve(kWsSplit, 2 << 20, stream(1));
}
static void reserve_without_memory() {
    g_oom = true;
    ws_reserve(kWsSplit, 1 << 20, stream(1));
}

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> all = {{"threads_on_one_stream", threads_on_one_stream},
                                                   {"another_stream_runs", another_stream_runs},
                                                   {"captures_have_their_own", captures_have_their_own},
                                                   {"graphs_give_back", graphs_give_back},
                                                   {"allocate_beside_a_capture", allocate_beside_a_capture},
                                                   {"capture_without_memory", capture_without_memory},
                                                   {"growth_frees", growth_frees},
                                                   {"without_memory", without_memory},
                                                   {"reserve_in_capture", reserve_in_capture},
                                                   {"reserve_without_memory", reserve_without_memory}};
    EXPECT(argc == 2 && all.count(argv[1]));
    all.at(argv[1])();
    printf("OK\n");
    return 0;
}
