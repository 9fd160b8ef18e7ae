// Library-owned workspaces of the prefill GEMMs (split-K partial sums, the W4A8 / W8A8 and fp16-accumulate
// pre-pass buffers), of the one-pass decode's tail (counters and part sums) and of the skinny kernel's slice sums, one
// buffer per (kind, device, stream).
//
// The reference keeps these buffers thread_local (src/kernels/gemm.cu:3258-3368), so two host threads never share
// one. Here the key is the stream a call is enqueued on: calls on one stream run in order, so they can share a
// buffer, while calls on two streams of one device (or two graphs replayed on two streams) get two buffers and cannot
// overwrite each other's data. A call's launches that write and read a buffer have to follow each other on the stream
// without another call's in between, and host threads may call on one stream (torch's threads share the default one),
// so a call holds the stream's lock (WsHold) from its first buffer to its last launch.
// A buffer grows on a call outside graph capture; the outgrown one is kept allocated
// (retired, never freed: a graph captured earlier may still read it). During capture a buffer that is too small is
// not grown: get returns nullptr and the caller either runs without it (the GEMM's split, the decode kernels; they
// do so too when the device has no memory left for it) or aborts with a message (the pre-passes), so callers size it
// first with an eager call or ws_reserve on that stream.
#include <map>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "qe_api.hpp"

namespace {
struct Ws {
    void* p = nullptr;
    size_t bytes = 0;
};
}  // namespace

struct StreamWs {
    std::mutex mu;  // held by WsHold; guards ws
    Ws ws[kNumWs];
};

namespace {
std::mutex g_mu;  // guards the containers below; never held while a stream's lock is waited for
std::map<std::pair<int, hipStream_t>, std::unique_ptr<StreamWs>> g_streams;  // (device, stream), never erased
std::vector<void*> g_retired;
int g_count[kNumWs];

StreamWs* stream_of(hipStream_t st) {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_mu);
    std::unique_ptr<StreamWs>& s = g_streams[std::make_pair(dev, st)];
    if (!s) s.reset(new StreamWs);
    return s.get();
}
}  // namespace

WsHold::WsHold(hipStream_t st) : st_(st), s_(stream_of(st)) { s_->mu.lock(); }
WsHold::~WsHold() { s_->mu.unlock(); }

void* WsHold::get(int kind, size_t bytes) {
    CHECK(kind >= 0 && kind < kNumWs, "workspace kind %d", kind);
    Ws& w = s_->ws[kind];
    if (w.bytes >= bytes) return w.p;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    HIP_CHECK(hipStreamIsCapturing(st_, &cs));
    if (cs != hipStreamCaptureStatusNone) return nullptr;
    void* np = nullptr;
    const hipError_t e = hipMalloc(&np, bytes);
    if (e == hipErrorOutOfMemory && kind != kWsI8 && kind != kWsH) {  // every other caller runs without its buffer
        (void)hipGetLastError();
        return nullptr;
    }
    HIP_CHECK(e);
    if (kind == kWsDec) {  // counters start at zero (the kernel sets them back to zero at the end of every call)
        HIP_CHECK(hipMemsetAsync(np, 0, bytes, st_));
        HIP_CHECK(hipStreamSynchronize(st_));
    }
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (w.p) g_retired.push_back(w.p);
        else g_count[kind]++;
    }
    w.p = np;
    w.bytes = bytes;
    return np;
}

size_t dec_tail_ctr_bytes() { return ((size_t)qe_num_cus() * 4 + 255) / 256 * 256; }

char* WsHold::dec_tail() {
    return static_cast<char*>(get(kWsDec, dec_tail_ctr_bytes() + (size_t)qe_num_cus() * 64 * 128 * 4));
}

void ws_reserve(int kind, size_t bytes, hipStream_t st) {
    if (bytes > 0) CHECK(WsHold(st).get(kind, bytes) != nullptr, "workspace reserve: called during graph capture");
}

int ws_count(int kind) {
    std::lock_guard<std::mutex> lk(g_mu);
    return kind >= 0 && kind < kNumWs ? g_count[kind] : 0;
}
