// SPDX-License-Identifier: Apache-2.0
// Host test of the scratch pool (csrc/kda_scratch.hip) against a model of the HIP runtime: streams
// whose work ends when the test says so, events, and an allocator that checks, each time a block is
// handed out again or freed, that every earlier use of it comes first in that stream's order. No GPU.
#include "kda_scratch.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

using namespace k3kda;

struct Stream {
    long issued = 0, done = 0;          // work items
    std::map<Stream *, long> after;     // what its next work is ordered behind
    bool blocking = true, capturing = false;
};
struct Event {
    Stream *s = nullptr;
    long seq = 0;
};
struct Alloc {
    size_t bytes;
    std::vector<std::pair<Stream *, long>> uses;
};

static Stream g_null;
static std::map<void *, Alloc> g_live;
struct Freed {
    Stream *s;
    size_t bytes;
    bool synced;
};
static std::vector<Freed> g_freed;          // with the runtime's pool until it is trimmed after a wait
static size_t g_bytes, g_limit = ~(size_t)0;
static int g_violations, g_null_in_capture, g_waits, g_refuse_wait, g_refuse_free, g_refuse_record, g_refuse_sync;
static std::vector<Stream *> g_streams;
static bool g_relaxed;

static Stream *S(hipStream_t st) { return st ? reinterpret_cast<Stream *>(st) : &g_null; }
static hipStream_t H(Stream *s) { return reinterpret_cast<hipStream_t>(s); }
static Stream *make(bool blocking)
{
    Stream *s = new Stream;
    s->blocking = blocking;
    g_streams.push_back(s);
    return s;
}
static bool before(Stream *s, long seq, Stream *by)   // work seq of s is over, or ordered before by's next
{
    if (s == by || s->done >= seq) return true;
    auto it = by->after.find(s);
    return it != by->after.end() && it->second >= seq;
}
// Work on the null stream waits for every blocking stream (and may not, while one is captured).
static void null_work(Stream *s)
{
    if (s != &g_null) return;
    for (Stream *o : g_streams)
        if (o->blocking) {
            if (o->capturing) g_null_in_capture++;
            s->after[o] = o->issued;
        }
}
static void launch(Stream *s, void *p)   // a kernel that uses p
{
    null_work(s);
    g_live.at(p).uses.push_back({s, ++s->issued});
}
static bool ordered(void *p, Stream *by)
{
    for (auto &u : g_live.at(p).uses)
        if (!before(u.first, u.second, by)) return false;
    return true;
}
static void finish(Stream *s) { s->done = s->issued; }

extern "C" {
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t st)
{
    null_work(S(st));
    size_t kept = 0;
    for (auto &f : g_freed) kept += f.bytes;
    if (g_bytes + kept + n > g_limit) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    g_live[*p] = Alloc{n, {}};
    g_bytes += n;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return hipMallocAsync(p, n, H(make(false))); }
hipError_t hipFreeAsync(void *p, hipStream_t st)
{
    if (g_refuse_free) return hipErrorInvalidValue;
    null_work(S(st));
    if (!ordered(p, S(st))) g_violations++;
    g_bytes -= g_live.at(p).bytes;
    g_freed.push_back({S(st), g_live.at(p).bytes, false});
    g_live.erase(p);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t st, hipStreamCaptureStatus *c)
{
    *c = S(st)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(new Event), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<Event *>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st)
{
    if (g_refuse_record) return hipErrorInvalidHandle;
    *reinterpret_cast<Event *>(e) = Event{S(st), S(st)->issued};
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e)
{
    if (!g_relaxed)
        for (Stream *s : g_streams)
            if (s->capturing) return hipErrorStreamCaptureUnsupported;
    Event *v = reinterpret_cast<Event *>(e);
    return v->s->done >= v->seq ? hipSuccess : hipErrorNotReady;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    Event *v = reinterpret_cast<Event *>(e);
    if (v->s->done < v->seq) v->s->done = v->seq;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t e, unsigned)
{
    if (g_refuse_wait) return hipErrorInvalidHandle;
    Event *v = reinterpret_cast<Event *>(e);
    null_work(S(st));
    if (v->s != S(st) && v->s->done < v->seq) g_waits++;
    long &a = S(st)->after[v->s];
    if (a < v->seq) a = v->seq;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st)
{
    if (g_refuse_sync) return hipErrorInvalidHandle;
    Stream *s = S(st);
    for (auto &a : s->after)
        if (a.first->done < a.second) a.first->done = a.second;
    finish(s);
    for (auto &f : g_freed) f.synced |= f.s == s;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned f) { return *st = H(make(f != hipStreamNonBlocking)), hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m)
{
    const bool was = g_relaxed;
    g_relaxed = *m == hipStreamCaptureModeRelaxed;
    *m = was ? hipStreamCaptureModeRelaxed : hipStreamCaptureModeGlobal;
    return hipSuccess;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t *p, int) { return *p = nullptr, hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t)
{
    std::vector<Freed> left;
    for (auto &f : g_freed)
        if (!f.synced) left.push_back(f);
    g_freed.swap(left);
    return hipSuccess;
}
}

static int g_failed;
#define CHECK(c) ((c) ? (void)0 : (void)(g_failed++, std::printf("  line %d: %s\n", __LINE__, #c)))

// A call on s with n bytes of scratch and one kernel; the block it had.
static void *call(Stream *s, size_t n, hipError_t *e = nullptr)
{
    StreamBuf b;
    const hipError_t r = scratch_alloc(b, n, s == &g_null ? nullptr : H(s));
    if (e) *e = r;
    if (r != hipSuccess) return nullptr;
    if (!ordered(b.p, s)) g_violations++;
    launch(s, b.p);
    return b.p;
}

constexpr size_t MB = 1ull << 20, GB = 1ull << 30;

static void reuse()
{
    Stream *a = make(false), *b = make(false);
    void *p = call(a, 10 * MB);
    CHECK(call(a, 9 * MB) == p);      // its own stream's
    CHECK(call(b, 9 * MB) != p);      // in flight: another
    finish(a);
    finish(b);
    void *q = call(&g_null, 9 * MB);
    CHECK(q == p || g_live.size() == 2);
    CHECK(g_waits == 0);
}

static void evict_leaves_blocks_in_flight()
{
    Stream *a = make(false), *b = make(false);
    call(a, 3 * GB);
    void *q = call(b, 3584 * MB);     // 6.5 GB: more than is kept, and a's block is in flight
    CHECK(g_waits == 0);              // nobody waits for a
    CHECK(!g_live.count(q));          // a plain allocation, freed with its call
    CHECK(g_bytes == 3 * GB);         // a's block is still there
    CHECK(g_null_in_capture == 0 && g_null.after.empty());
}

static void evict_idle_blocks_on_the_calls_stream()
{
    Stream *a = make(false), *b = make(false), *c = make(true);
    call(a, 3 * GB);
    finish(a);
    c->capturing = true;              // a blocking stream's capture: no null-stream work now
    call(b, 3584 * MB);
    CHECK(g_bytes == 3584 * MB);
    CHECK(g_null_in_capture == 0 && g_null.after.empty());
    c->capturing = false;
}

static void evict_own_block_in_flight()
{
    Stream *a = make(false);
    call(a, 3 * GB);
    call(a, 3584 * MB);               // in order on the same stream
    CHECK(g_bytes == 3584 * MB);
}

static void refused_wait()
{
    Stream *a = make(false), *b = make(false);
    call(a, 3 * GB);
    finish(a);
    g_refuse_wait = 1;
    call(b, 3584 * MB);               // may neither take nor free a's block
    CHECK(g_bytes == 3 * GB);
    call(b, 1 * GB);
    g_refuse_wait = 0;
    CHECK(g_bytes >= 3 * GB);
}

static void refused_free()
{
    Stream *a = make(false);
    void *p = call(a, 3 * GB);
    finish(a);
    g_refuse_free = 1;
    {
        StreamBuf b;                  // 3.5 GB more than is kept: plain, or none
        CHECK(scratch_alloc(b, 3584 * MB, H(a)) == hipSuccess);
        g_refuse_free = 0;
    }
    CHECK(g_bytes == 3 * GB);         // still counted ...
    CHECK(call(a, 3 * GB) == p);      // ... and still whole
}

static void refused_record()
{
    Stream *a = make(false), *b = make(false);
    g_refuse_record = 1;
    void *p = call(a, 10 * MB);       // the host waits
    CHECK(a->done == a->issued);
    CHECK(call(b, 10 * MB) == p);
    g_refuse_sync = 1;
    call(b, 10 * MB);                 // its end cannot be known: never lent again
    g_refuse_record = g_refuse_sync = 0;
    CHECK(call(b, 10 * MB) != p);
    CHECK(call(a, 10 * MB) != p);
}

static void last_release()
{
    Stream *a = make(false);
    call(a, 10 * MB);                 // in flight
    call(&g_null, 20 * MB);
    StreamBuf *b = new StreamBuf;
    CHECK(scratch_alloc(*b, 30 * MB, H(a)) == hipSuccess);
    launch(a, b->p);
    ws_handles(-1);
    CHECK(g_bytes >= 30 * MB && g_bytes < 40 * MB);   // the busy one
    CHECK(g_null.after.find(a) == g_null.after.end());   // the null stream did not wait for a
    delete b;
    CHECK(g_bytes == 0);
    ws_handles(1);
}

static void capture()
{
    Stream *a = make(false), *b = make(false);
    call(b, 10 * MB);
    finish(b);
    a->capturing = true;
    void *p = call(a, 10 * MB);       // the graph's own
    CHECK(!g_live.count(p));
    void *q = call(b, 10 * MB), *r = call(&g_null, 10 * MB);
    CHECK(g_live.count(q) && g_live.count(r));
    a->capturing = false;
}

static void out_of_memory()
{
    Stream *a = make(false), *b = make(false), *c = make(false);
    hipError_t e;
    g_limit = 1000 * MB;
    call(a, 256 * MB);                // held, in flight
    call(&g_null, 256 * MB);          // the null stream's: not touched from another
    void *held = nullptr;
    {
        StreamBuf busy;
        CHECK(scratch_alloc(busy, 128 * MB, H(c)) == hipSuccess);
        launch(c, held = busy.p);
        call(b, 600 * MB, &e);        // fits without the idle 256
        CHECK(e == hipSuccess && g_live.count(held));
        call(b, 900 * MB, &e);        // does not fit
        CHECK(e == hipErrorOutOfMemory && g_live.count(held));
    }
    (void)hipStreamSynchronize(H(b)); // the 600 MB of b's plain call
    call(&g_null, 1000 * MB, &e);     // without everything idle, the null stream's own too
    CHECK(e == hipSuccess);
    g_limit = 2000 * MB;
    call(a, 512 * MB);
    void *w = nullptr;
    CHECK(device_alloc(&w, 1900 * MB) == hipSuccess);   // weights
    CHECK(device_alloc(&w, 1900 * MB) == hipErrorOutOfMemory && !w);
}

static void out_of_memory_under_capture()
{
    Stream *a = make(false), *b = make(false);
    hipError_t e;
    g_limit = 1000 * MB;
    call(a, 512 * MB);
    b->capturing = true;
    call(b, 600 * MB, &e);            // the graph's allocation: nothing is waited for
    CHECK(e == hipErrorOutOfMemory && a->done < a->issued);
    b->capturing = false;
}

int main(int argc, char **argv)
{
    struct { const char *name; void (*run)(); } tests[] = {
        {"reuse", reuse}, {"evict_leaves_blocks_in_flight", evict_leaves_blocks_in_flight},
        {"evict_idle_blocks_on_the_calls_stream", evict_idle_blocks_on_the_calls_stream},
        {"evict_own_block_in_flight", evict_own_block_in_flight}, {"refused_wait", refused_wait},
        {"refused_free", refused_free}, {"refused_record", refused_record}, {"last_release", last_release},
        {"capture", capture}, {"out_of_memory", out_of_memory}, {"out_of_memory_under_capture", out_of_memory_under_capture},
    };
    if (argc < 2) {
        for (auto &t : tests) std::printf("%s\n", t.name);
        return 0;
    }
    for (auto &t : tests)
        if (!std::strcmp(argv[1], t.name)) {
            ws_handles(1);
            t.run();
            for (Stream *s : g_streams) finish(s);
            finish(&g_null);
            ws_handles(-1);
            CHECK(g_violations == 0);
            return g_failed != 0;
        }
    return 2;
}
