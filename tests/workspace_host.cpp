// Host model of the HIP calls that qengine_amd/csrc/workspace.cpp makes, and the scenarios of test_workspace.py on it:
// linked with workspace.cpp by g++, no GPU and no HIP runtime. "Device memory" is malloc; a scenario sets what a stream's
// capture status is and which calls fail.
#include <atomic>
#include <chrono>
#include <cstring>
#include <map>
#include <set>
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
std::set<void*> g_live;  // allocations not freed
}  // namespace

// ---- the HIP calls ----
extern "C" {
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "model"; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    *p = malloc(n);
    g_live.insert(*p);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
    memset(p, v, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
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

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> all = {{"threads_on_one_stream", threads_on_one_stream},
                                                   {"another_stream_runs", another_stream_runs}};
    EXPECT(argc == 2 && all.count(argv[1]));
    all.at(argv[1])();
    printf("OK\n");
    return 0;
}
