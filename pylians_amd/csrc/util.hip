// Error reporting, zero-fill and library-owned workspaces.
#include <stdarg.h>

#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "common.hpp"
#include "util.hpp"

namespace pyl {

static thread_local char g_err[1024] = "";

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}
const char* last_error() { return g_err; }

// Zero-fill with a kernel rather than hipMemsetAsync, so that the clear is an ordinary kernel
// node when a caller captures the stream into a graph.
__device__ __forceinline__ void zero_body(uint4* __restrict__ p, long long n16, unsigned char* __restrict__ tail,
                                          int ntail) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
        p[i] = make_uint4(0u, 0u, 0u, 0u);
    if (blockIdx.x == 0 && (int)threadIdx.x < ntail) tail[threadIdx.x] = 0;
}
__global__ void k_zero(uint4* __restrict__ p, long long n16, unsigned char* __restrict__ tail, int ntail) {
    zero_body(p, n16, tail, ntail);
}
// batched: buffer blockIdx.y of the table (16-byte aligned pointer, byte count)
__global__ void k_zero_b(const ZeroArgs* __restrict__ tab) {
    const ZeroArgs z = tab[blockIdx.y];
    const long long n16 = (long long)(z.bytes / 16);
    zero_body((uint4*)z.ptr, n16, (unsigned char*)z.ptr + n16 * 16, (int)(z.bytes % 16));
}

int zero_fill(void* ptr, size_t bytes, hipStream_t st) {
    if (!bytes) return OK;
    PYL_CHECK(((uintptr_t)ptr & 15) == 0, E_ARG, "zero_fill needs 16-byte alignment");
    const long long n16 = (long long)(bytes / 16);
    const int ntail = (int)(bytes % 16);
    long long blocks = (n16 + 255) / 256;
    if (blocks > 16384) blocks = 16384;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, st, (uint4*)ptr, n16,
                       (unsigned char*)ptr + n16 * 16, ntail);
    PYL_HIP(hipGetLastError());
    return OK;
}

__global__ __launch_bounds__(1024) void k_sum_parts(const double* __restrict__ part, int nb, double* __restrict__ out) {
    __shared__ double red[16];
    const int tid = threadIdx.x;
    double a = 0.0;
    for (int b = tid; b < nb; b += 1024) a += part[b];
    for (int off = 32; off > 0; off >>= 1) a += __shfl_down(a, off, 64);
    if ((tid & 63) == 0) red[tid >> 6] = a;
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int w = 0; w < 16; ++w) s += red[w];
        out[0] = s;
    }
}

int sum_parts(const double* part, int nb, double* out, hipStream_t st) {
    hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(1024), 0, st, part, nb, out);
    PYL_HIP(hipGetLastError());
    return OK;
}

// Grow-only device buffers keyed by (device, slot).  Growing synchronises the device before
// freeing the old buffer, so work already queued on it finishes first.
struct WsArena {
    int dev = 0;
    bool sealed = false;
    std::map<int, std::pair<void*, size_t>> slots;
    // fixed arena: every slot and table is carved from [base, base + cap) in request order
    char* base = nullptr;
    size_t cap = 0, used = 0;
    hipStream_t st = nullptr;   // fixed arena: of its uploads; a stream's set: the stream in a StreamScope
    bool of_stream = false;     // a stream's set: all that used its buffers is on st or ordered before it
};
static thread_local WsArena* t_arena = nullptr;

static void* carve(WsArena* a, size_t bytes, int* rc) {
    const size_t at = (a->used + 255) / 256 * 256;
    if (at > a->cap || bytes > a->cap - at) {
        set_error("scratch of %zu bytes exhausted: this call needs more than %zu bytes (a larger grid than the "
                  "no-allocation entry point supports)", a->cap, at + bytes);
        *rc = E_ALLOC;
        return nullptr;
    }
    a->used = at + bytes;
    return a->base + at;
}

hipError_t device_alloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        stream_ws_release(false);
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

// frees a buffer once the work that may use it is done; a buffer that cannot be freed is kept
static bool give_back(std::pair<void*, size_t>& e, int* rc, const WsArena* a) {
    if (!e.first) return true;
    const hipError_t w = a && a->of_stream ? hipStreamSynchronize(a->st) : hipDeviceSynchronize();
    if (w != hipSuccess || hipFree(e.first) != hipSuccess) {
        (void)hipGetLastError();
        set_error("a workspace in use could not be freed");
        *rc = E_ALLOC;
        return false;
    }
    e = std::make_pair(nullptr, (size_t)0);
    return true;
}

static void* grow(std::pair<void*, size_t>& e, size_t bytes, int* rc, const WsArena* a = nullptr) {
    if (!give_back(e, rc, a)) return nullptr;
    size_t want = bytes < 256 ? 256 : bytes;
    if (device_alloc(&e.first, want) != hipSuccess) {
        e.first = nullptr;
        set_error("workspace allocation of %zu bytes failed", want);
        *rc = E_ALLOC;
        return nullptr;
    }
    e.second = want;
    return e.first;
}

static std::mutex g_ws_mu;
static std::map<std::pair<int, int>, std::pair<void*, size_t>>& shared_ws() {
    static auto* m = new std::map<std::pair<int, int>, std::pair<void*, size_t>>();   // outlives every caller
    return *m;
}

void workspace_drop(int slot) {
    int rc = OK, dev = 0;
    if (WsArena* a = t_arena) {
        if (!a->base && !a->sealed) give_back(a->slots[slot], &rc, a);
        return;
    }
    if (hipGetDevice(&dev) != hipSuccess) return;
    std::lock_guard<std::mutex> lk(g_ws_mu);
    give_back(shared_ws()[std::make_pair(dev, slot)], &rc, nullptr);
}

void* workspace(int slot, size_t bytes, int* rc) {
    *rc = OK;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        set_error("hipGetDevice failed");
        *rc = E_LAUNCH;
        return nullptr;
    }
    if (WsArena* a = t_arena) {
        if (a->dev != dev) {
            set_error("graph workspace of device %d used on device %d", a->dev, dev);
            *rc = E_ARG;
            return nullptr;
        }
        auto& e = a->slots[slot];
        if (e.second >= bytes && e.first) return e.first;
        if (a->base) {
            void* p = carve(a, bytes, rc);
            if (p) e = std::make_pair(p, bytes);
            return p;
        }
        if (a->sealed) {
            set_error("graph workspace slot %d would grow from %zu to %zu bytes during capture", slot, e.second,
                      bytes);
            *rc = E_ALLOC;
            return nullptr;
        }
        return grow(e, bytes, rc, a);
    }
    std::lock_guard<std::mutex> lk(g_ws_mu);
    auto& e = shared_ws()[std::make_pair(dev, slot)];
    if (e.second >= bytes && e.first) return e.first;
    return grow(e, bytes, rc);
}

void* host_pinned(size_t bytes, int* rc) {
    static std::mutex mu;
    static std::map<int, std::pair<void*, size_t>> bufs;
    *rc = OK;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        set_error("hipGetDevice failed");
        *rc = E_LAUNCH;
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(mu);
    auto& e = bufs[dev];
    if (e.first && e.second >= bytes) return e.first;
    if (e.first) {
        (void)hipDeviceSynchronize();
        (void)hipHostFree(e.first);
        e = std::make_pair(nullptr, (size_t)0);
    }
    const size_t want = bytes < 4096 ? 4096 : bytes;
    if (hipHostMalloc(&e.first, want, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        e.first = nullptr;
        set_error("pinned host allocation of %zu bytes failed", want);
        *rc = E_ALLOC;
        return nullptr;
    }
    e.second = want;
    return e.first;
}

WsArena* ws_arena_create() {
    WsArena* a = new WsArena();
    if (hipGetDevice(&a->dev) != hipSuccess) a->dev = 0;
    return a;
}

WsArena* ws_arena_fixed(void* base, size_t cap) {
    WsArena* a = ws_arena_create();
    a->base = (char*)base;
    a->cap = cap;
    return a;
}

void ws_arena_fixed_reset(WsArena* a, hipStream_t st) {
    a->slots.clear();
    a->used = 0;
    a->st = st;
}

bool arena_fixed() { return t_arena && t_arena->base; }

void* arena_upload(const void* host, size_t bytes, int* rc) {
    *rc = OK;
    WsArena* a = t_arena;
    if (!a || !a->base) {
        set_error("arena_upload outside a fixed arena");
        *rc = E_ARG;
        return nullptr;
    }
    void* p = carve(a, bytes, rc);
    if (!p) return nullptr;
    if (hipMemcpyAsync(p, host, bytes, hipMemcpyHostToDevice, a->st) != hipSuccess) {
        set_error("table upload into the scratch failed");
        *rc = E_LAUNCH;
        return nullptr;
    }
    return p;
}

void ws_arena_seal(WsArena* a) {
    if (a) a->sealed = true;
}

void ws_arena_destroy(WsArena* a) {
    if (!a) return;
    if (a->base) {   // fixed arenas own no memory
        delete a;
        return;
    }
    int cur = 0;
    (void)hipGetDevice(&cur);
    (void)hipSetDevice(a->dev);
    (void)hipDeviceSynchronize();
    for (auto& kv : a->slots)
        if (kv.second.first) (void)hipFree(kv.second.first);
    (void)hipSetDevice(cur);
    delete a;
}

size_t ws_arena_bytes(const WsArena* a) {
    size_t s = 0;
    if (a)
        for (auto& kv : a->slots) s += kv.second.second;
    return s;
}

// Workspaces of the deposits that may run on several streams at once (StreamScope): at most STREAM_WS sets a device.  A
// further stream takes over the set used longest ago: nothing is freed and the host does not wait, its kernels run
// behind the event of that set's last call.  A stream's own calls run in order and need no event (it costs a call of
// 87 us 4.6), and a handle comes back only after its work (hipStreamDestroy waits for it), so the handle names the queue --
// except hipStreamPerThread, which is another queue in every thread: there the thread counts too, and as a
// thread's id may come back as well, its calls always have the event.
constexpr size_t STREAM_WS = 4;
struct Queue {
    hipStream_t st;
    std::thread::id owner;   // hipStreamPerThread: the thread that passed it
    explicit Queue(hipStream_t s) : st(s) {
        if (s == hipStreamPerThread) owner = std::this_thread::get_id();
    }
    bool operator==(const Queue& o) const { return st == o.st && owner == o.owner; }
};
struct StreamWs {
    int dev;
    Queue q;                     // whose set it is (under the pool's mutex)
    std::mutex mu;               // held while a call queues its kernels; guards what follows
    WsArena* arena;
    Queue last;                  // queue of the last call
    enum { FREE, OPEN, MARKED } state = FREE;   // no call; a call without an event behind it; with
    hipEvent_t done = nullptr;
    StreamWs(int d, const Queue& k) : dev(d), q(k), arena(ws_arena_create()), last(k) { arena->of_stream = true; }
    ~StreamWs() {
        ws_arena_destroy(arena);
        if (done) (void)hipEventDestroy(done);
    }
};

namespace {
struct StreamPool {
    std::mutex mu;
    std::vector<std::shared_ptr<StreamWs>> sets;   // in the order of their last use
};
StreamPool& stream_pool() {
    static StreamPool* p = new StreamPool();   // outlives every caller
    return *p;
}
}  // namespace

// the set of a queue; shared: whether another queue has one too (and may take this one over)
static std::shared_ptr<StreamWs> stream_ws(hipStream_t st, bool* shared) {
    StreamPool& P = stream_pool();
    int dev = 0;
    (void)hipGetDevice(&dev);
    const Queue q(st);
    std::lock_guard<std::mutex> lk(P.mu);
    size_t n = 0, oldest = P.sets.size(), own = P.sets.size();
    for (size_t i = P.sets.size(); i-- > 0;) {
        if (P.sets[i]->dev != dev) continue;
        ++n;
        oldest = i;
        if (P.sets[i]->q == q) own = i;
    }
    if (own == P.sets.size() && n >= STREAM_WS) {
        own = oldest;
        P.sets[own]->q = q;
    }
    std::shared_ptr<StreamWs> w;
    if (own < P.sets.size()) {
        w = P.sets[own];
        P.sets.erase(P.sets.begin() + (long)own);
    } else {
        w = std::make_shared<StreamWs>(dev, q);
        ++n;
    }
    P.sets.push_back(w);
    *shared = n > 1;
    return w;
}

void stream_ws_release(bool all) {
    std::vector<std::shared_ptr<StreamWs>> out;   // freed after the lock is given back; a set in use, by its last user
    StreamPool& P = stream_pool();
    std::lock_guard<std::mutex> lk(P.mu);
    for (size_t i = P.sets.size(); i-- > 0;)
        if (all || P.sets[i].use_count() == 1) {
            out.push_back(P.sets[i]);
            P.sets.erase(P.sets.begin() + (long)i);
        }
}

StreamScope::StreamScope(hipStream_t s) : st(s) {
    if (t_arena) return;   // a graph's or a fixed arena: that one
    // another stream may be capturing: these calls touch nothing of its graph, and would end its capture otherwise
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    ws = stream_ws(st, &mark);
    mark = mark || st == hipStreamPerThread;
    ws->mu.lock();
    const Queue q(st);
    hipError_t e = hipSuccess;
    if (mark && !ws->done) e = hipEventCreateWithFlags(&ws->done, hipEventDisableTiming);
    if (e == hipSuccess && ws->state != StreamWs::FREE && (!(ws->last == q) || st == hipStreamPerThread))
        // OPEN: the only set of its time when it was used last; the first to take it over waits
        e = ws->state == StreamWs::MARKED ? hipStreamWaitEvent(st, ws->done, 0) : hipDeviceSynchronize();
    if (e != hipSuccess) {
        (void)hipGetLastError();
        ws->mu.unlock();
        ws.reset();
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        ok = false;
        return;
    }
    ws->last = q;
    ws->arena->st = st;
    t_arena = ws->arena;
}
StreamScope::~StreamScope() {
    if (!ws) return;
    t_arena = nullptr;
    ws->state = StreamWs::OPEN;
    if (mark) {
        if (hipEventRecord(ws->done, st) == hipSuccess) {
            ws->state = StreamWs::MARKED;
        } else {   // nothing to order the next call behind: wait here
            (void)hipGetLastError();
            if (hipStreamSynchronize(st) == hipSuccess) ws->state = StreamWs::FREE;
        }
    }
    ws->mu.unlock();
    ws.reset();
    (void)hipThreadExchangeStreamCaptureMode(&mode);
}

ArenaScope::ArenaScope(WsArena* a) : prev(t_arena) { t_arena = a; }
ArenaScope::~ArenaScope() { t_arena = prev; }

constexpr size_t PINNED_KEPT = 4;
static std::mutex g_pin_mu;
static std::vector<std::pair<void*, size_t>>& pin_free() {
    static auto* v = new std::vector<std::pair<void*, size_t>>();   // outlives every caller
    return *v;
}

int PinnedScope::take(size_t want) {
    {
        std::lock_guard<std::mutex> lk(g_pin_mu);
        auto& v = pin_free();
        for (size_t i = 0; i < v.size(); ++i)
            if (v[i].second >= want) {
                p = v[i].first;
                bytes = v[i].second;
                v.erase(v.begin() + (long)i);
                return OK;
            }
    }
    size_t b = 1 << 16;
    while (b < want) b *= 2;
    if (hipHostMalloc(&p, b, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        p = nullptr;
        set_error("pinned host allocation of %zu bytes failed", b);
        return E_ALLOC;
    }
    bytes = b;
    return OK;
}

void pinned_release() {
    std::vector<std::pair<void*, size_t>> out;
    {
        std::lock_guard<std::mutex> lk(g_pin_mu);
        out.swap(pin_free());
    }
    for (auto& e : out) (void)hipHostFree(e.first);
}

PinnedScope::~PinnedScope() {
    if (!p) return;
    {
        std::lock_guard<std::mutex> lk(g_pin_mu);
        auto& v = pin_free();
        if (v.size() < PINNED_KEPT) {
            v.emplace_back(p, bytes);
            return;
        }
        for (auto& e : v)   // the larger one stays
            if (e.second < bytes) {
                std::swap(e.first, p);
                std::swap(e.second, bytes);
                break;
            }
    }
    (void)hipHostFree(p);
}

}  // namespace pyl
