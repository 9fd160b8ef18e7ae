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
// A buffer grows on a call outside graph capture; the outgrown one is freed when the stream's work on it is done.
//
// Calls under graph capture never get the stream's buffer: a graph replays on whatever stream it is launched on, beside
// eager calls on the stream it was captured on or another graph captured there. The calls of one capture on one stream
// share buffers of their own, which the graph holds (a user object that it and the executables made of it retain) and
// which return to a pool, for later captures, when the last of these is destroyed. So the pool is as large as the graphs
// that lived at one time needed. The pre-passes and the GEMM's split keep the rule that a capture needs its stream
// sized first (an eager call or ws_reserve there): get returns nullptr else, and the caller runs without the buffer (the
// split) or aborts with a message (the pre-passes). The decode kernels' buffers need no preparation. They and the split
// also run without a buffer when the device has no memory left for it; a failed hipMalloc takes longer than the call,
// so the next kRetry calls do not try again.
#include <map>
#include <memory>
#include <mutex>
#include <utility>

#include "qe_api.hpp"

namespace {
constexpr int kRetry = 256;  // calls that do without a buffer after the device had no memory for it, before it is asked again
struct Ws {
    void* p = nullptr;
    size_t bytes = 0;
    size_t refused = 0;  // the size it had no memory for, and the calls of at least that size left to do without
    int wait = 0;
};
struct CapBuf {  // a buffer that a graph holds, or one in the pool (owner 0)
    int dev, kind;
    void* p;
    size_t bytes;
    unsigned long long owner;  // the capture's id; guarded by State::mu
};
}  // namespace

struct StreamWs {
    int dev = 0;
    std::mutex mu;  // held by WsHold; guards the rest
    Ws ws[kNumWs];
    CapBuf* cap[kNumWs] = {};  // of the stream's last capture
};

namespace {
struct State {
    std::mutex mu;  // guards the rest; never held over a HIP call or while a stream's lock is waited for
    std::map<std::pair<int, hipStream_t>, std::unique_ptr<StreamWs>> streams;  // (device, stream), never erased
    std::multimap<std::pair<int, int>, CapBuf*> pool;  // (device, kind)
    int count[kNumWs] = {};
};
State& state() {  // never destroyed: graphs may outlive static objects
    static State* s = new State;
    return *s;
}

StreamWs* stream_of(hipStream_t st) {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(state().mu);
    std::unique_ptr<StreamWs>& s = state().streams[std::make_pair(dev, st)];
    if (!s) {
        s.reset(new StreamWs);
        s->dev = dev;
    }
    return s.get();
}

// whether st is being captured, the capture's id and its graph. (The legacy default stream cannot be captured.)
bool capturing(hipStream_t st, unsigned long long* id, hipGraph_t* graph) {
    if (st == nullptr) return false;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    HIP_CHECK(hipStreamGetCaptureInfo_v2(st, &cs, id, graph, nullptr, nullptr));
    return cs != hipStreamCaptureStatusNone;
}

// counters start at zero (the kernel sets them back to zero at the end of every call); on a stream of its own, as st may
// be in a capture
void zero_fill(void* p, size_t bytes) {
    hipStream_t s = nullptr;
    HIP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    HIP_CHECK(hipMemsetAsync(p, 0, bytes, s));
    HIP_CHECK(hipStreamSynchronize(s));
    HIP_CHECK(hipStreamDestroy(s));
}

// the last graph or executable that holds the buffer is gone (called by the HIP runtime: no HIP calls in here)
void give_back(void* arg) {
    CapBuf* b = static_cast<CapBuf*>(arg);
    std::lock_guard<std::mutex> lk(state().mu);
    b->owner = 0;
    state().count[b->kind]--;
    state().pool.emplace(std::make_pair(b->dev, b->kind), b);
}

// device memory inside a capture or beside one of another thread, which the default (global) mode forbids: the allocation
// is not part of any graph, so this thread leaves that mode for it
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { HIP_CHECK(hipThreadExchangeStreamCaptureMode(&mode)); }
    ~RelaxedCapture() { HIP_CHECK(hipThreadExchangeStreamCaptureMode(&mode)); }
};

// the smallest pooled buffer of at least `bytes`, else a new one (sizes in four steps per octave, so that few suffice for
// captures of many shapes); nullptr when the device has no memory for it
CapBuf* take(int dev, int kind, size_t bytes, unsigned long long id) {
    State& st = state();
    {
        std::lock_guard<std::mutex> lk(st.mu);
        auto r = st.pool.equal_range(std::make_pair(dev, kind));
        auto best = r.second;
        for (auto it = r.first; it != r.second; ++it)
            if (it->second->bytes >= bytes && (best == r.second || it->second->bytes < best->second->bytes)) best = it;
        if (best != r.second) {
            CapBuf* b = best->second;
            st.pool.erase(best);
            b->owner = id;
            st.count[kind]++;
            return b;
        }
    }
    size_t step = 1 << 18;
    while (step * 8 <= bytes) step *= 2;
    bytes = (bytes + step - 1) / step * step;
    RelaxedCapture relaxed;
    void* p = nullptr;
    const hipError_t e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        return nullptr;
    }
    HIP_CHECK(e);
    if (kind == kWsDec) zero_fill(p, bytes);
    std::lock_guard<std::mutex> lk(st.mu);
    st.count[kind]++;
    return new CapBuf{dev, kind, p, bytes, id};
}

void* capture_buf(StreamWs* s, int kind, size_t bytes, unsigned long long id, hipGraph_t graph) {
    CapBuf* b = s->cap[kind];
    if (b) {
        std::lock_guard<std::mutex> lk(state().mu);
        if (b->owner == id && b->bytes >= bytes) return b->p;
    }
    b = take(s->dev, kind, bytes, id);
    if (!b) return nullptr;
    hipUserObject_t o = nullptr;
    HIP_CHECK(hipUserObjectCreate(&o, b, give_back, 1, hipUserObjectNoDestructorSync));
    HIP_CHECK(hipGraphRetainUserObject(graph, o, 1, hipGraphUserObjectMove));
    s->cap[kind] = b;
    return b->p;
}

bool needs_sizing(int kind) { return kind == kWsSplit || kind == kWsI8 || kind == kWsH; }
}  // namespace

WsHold::WsHold(hipStream_t st) : st_(st), s_(stream_of(st)) { s_->mu.lock(); }
WsHold::~WsHold() { s_->mu.unlock(); }

void* WsHold::get(int kind, size_t bytes, bool retry) {
    CHECK(kind >= 0 && kind < kNumWs, "workspace kind %d", kind);
    Ws& w = s_->ws[kind];
    unsigned long long id = 0;
    hipGraph_t graph = nullptr;
    if (capturing(st_, &id, &graph)) return needs_sizing(kind) && w.bytes < bytes ? nullptr : capture_buf(s_, kind, bytes, id, graph);
    if (w.bytes >= bytes) return w.p;
    const bool optional = kind != kWsI8 && kind != kWsH;  // the caller runs without it
    if (optional && !retry && w.wait > 0 && bytes >= w.refused) {
        w.wait--;
        return nullptr;
    }
    RelaxedCapture relaxed;
    void* np = nullptr;
    const hipError_t e = hipMalloc(&np, bytes);
    if (e == hipErrorOutOfMemory && optional) {
        (void)hipGetLastError();
        w.refused = bytes;
        w.wait = kRetry;
        return nullptr;
    }
    HIP_CHECK(e);
    if (kind == kWsDec) zero_fill(np, bytes);
    if (w.p) {  // only this stream's calls use it, and they are all enqueued (the lock)
        HIP_CHECK(hipStreamSynchronize(st_));
        HIP_CHECK(hipFree(w.p));
    } else {
        std::lock_guard<std::mutex> lk(state().mu);
        state().count[kind]++;
    }
    w.p = np;
    w.bytes = bytes;
    w.wait = 0;
    return np;
}

size_t WsHold::sized(int kind) const { return s_->ws[kind].bytes; }

size_t dec_tail_ctr_bytes() { return ((size_t)qe_num_cus() * 4 + 255) / 256 * 256; }

char* WsHold::dec_tail() {
    return static_cast<char*>(get(kWsDec, dec_tail_ctr_bytes() + (size_t)qe_num_cus() * 64 * 128 * 4));
}

void ws_reserve(int kind, size_t bytes, hipStream_t st) {
    if (bytes == 0) return;
    unsigned long long id = 0;
    hipGraph_t graph = nullptr;
    WsHold hold(st);
    if (capturing(st, &id, &graph)) CHECK(hold.sized(kind) >= bytes, "workspace reserve: called during graph capture");
    else CHECK(hold.get(kind, bytes, true) != nullptr, "workspace reserve: no memory for %zu bytes", bytes);
}

int ws_count(int kind) {
    std::lock_guard<std::mutex> lk(state().mu);
    return kind >= 0 && kind < kNumWs ? state().count[kind] : 0;
}
