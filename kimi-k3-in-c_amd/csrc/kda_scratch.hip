// SPDX-License-Identifier: Apache-2.0
// kda_scratch.hip - scratch blocks kept between calls (host code only; no counterpart in the
// reference, whose scratch is the caller's).
//
// Blocks are kept while any weight set is uploaded (handles > 0), since hipMallocAsync +
// hipFreeAsync cost the host 10-11 us a pair, and after a synchronisation, when the runtime's
// pool has given its memory back, 50 us for 64 MB and ~350 us for the 1.4 GB of an 8192-token
// layer; a kept block costs ~1 us.
//  * A block is handed to one call at a time (busy). Its next call is on the same stream, so
//    stream order protects it, or the block is idle by its event.
//  * The legacy null stream lives for ever, so equality of the handle is identity and no event
//    is needed. Any other stream may be destroyed and its handle given to a new one: its blocks
//    carry an event recorded after the call's last launch, waited for on reuse.
//  * No call waits for another stream's block: it gets a new one while the device's blocks
//    stay within WS_KEEP_BYTES, and past that a plain stream allocation. Blocks too small for the
//    call that are its stream's own or idle are given back first, on the call's stream.
//  * A block leaves the list only when the runtime has taken it back; where the wait for its last
//    call or the free is refused it stays listed, counted and whole.
//  * Calls being captured into a graph take plain stream allocations (the graph's own nodes).
//  * Where an allocation fails, idle memory of the pool's must not be the reason: every block that
//    no call holds goes back, the host waits for that, and the allocation is tried again.
//  * The last release gives every block back: the null stream's on it, any other on a stream of
//    this file's own behind its event, so no stream of the caller's waits. A block whose call is
//    still being issued then goes back with that call.
#include "kda_scratch.h"

#include <mutex>
#include <vector>

namespace k3kda {

constexpr size_t WS_KEEP_BYTES = 4ull << 30;   // per device, of 288 GB
constexpr size_t WS_MIN_BLOCK = 1u << 20;
constexpr int WS_MAX_DEV = 64;

struct WsBlock {
    void *p;
    size_t size;
    int dev;
    hipStream_t last;   // stream of its last call
    hipEvent_t ev;      // after that call; none for the null stream
    bool busy;
    bool idle;          // no work is left on it and no event says so (the host has waited)
};

namespace {

struct WsPool {
    std::mutex mu;
    std::vector<WsBlock *> blocks;       // all of them, busy ones too
    size_t held[WS_MAX_DEV] = {};        // bytes per device
    hipStream_t own[WS_MAX_DEV] = {};    // for the last release
    int handles = 0;
};

WsPool &ws_pool()
{
    static WsPool *p = new WsPool;   // never destroyed: calls may outlive static destructors
    return *p;
}

// Sizes in steps of a quarter of a power of two, so that slowly growing requests share blocks.
size_t ws_class(size_t bytes)
{
    if (bytes <= WS_MIN_BLOCK) return WS_MIN_BLOCK;
    size_t step = WS_MIN_BLOCK / 4;
    while (step * 8 < bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

bool ok(hipError_t e)
{
    if (e == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
}

// Event queries are kept out of the rules of a capture that another stream or thread may have
// open in its global mode.
struct RelaxedCapture {
    hipStreamCaptureMode m = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&m); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&m); }
};

struct OnDevice {
    int was = -1;
    bool good;
    explicit OnDevice(int dev)
    {
        int cur = 0;
        good = ok(hipGetDevice(&cur));
        if (good && cur != dev) {
            good = ok(hipSetDevice(dev));
            if (good) was = cur;
        }
    }
    ~OnDevice()
    {
        if (was >= 0) (void)ok(hipSetDevice(was));
    }
};

// The block's last call is over or on st itself: st need not wait to use or free it.
bool ws_ready(const WsBlock *k, hipStream_t st)
{
    return k->idle || k->last == st || (k->ev && ok(hipEventQuery(k->ev)));
}

// What st does next comes after the block's last call.
bool ws_order(const WsBlock *k, hipStream_t st)
{
    if (k->idle) return true;
    return k->ev ? ok(hipStreamWaitEvent(st, k->ev, 0)) : k->last == st;
}

// Give block i back to the runtime in st's order. False: refused, the block stays.
bool ws_give(WsPool &P, size_t i, hipStream_t st)
{
    WsBlock *k = P.blocks[i];
    if (!ws_order(k, st) || !ok(hipFreeAsync(k->p, st))) return false;
    if (k->ev) (void)ok(hipEventDestroy(k->ev));
    P.held[k->dev] -= k->size;
    delete k;
    P.blocks.erase(P.blocks.begin() + (long)i);
    return true;
}

// This file's own stream on a device: non-blocking, so the null stream and the caller's do not
// wait for it, nor it for them. Null where it cannot be made.
hipStream_t ws_own_stream(WsPool &P, int dev)
{
    if (!P.own[dev]) {
        OnDevice d(dev);
        if (!d.good || !ok(hipStreamCreateWithFlags(&P.own[dev], hipStreamNonBlocking))) P.own[dev] = nullptr;
    }
    return P.own[dev];
}

// Give back every block that no call holds, of one device or (-1) of all; blocks of the null
// stream only with null_too, since that is work on it. The number given back.
int ws_give_all(WsPool &P, int dev, bool null_too)
{
    RelaxedCapture relaxed;
    int n = 0;
    for (size_t i = P.blocks.size(); i-- > 0;) {
        const WsBlock *k = P.blocks[i];
        if (k->busy || (dev >= 0 && k->dev != dev)) continue;
        if (k->last == nullptr) {   // in the null stream's order, on its device
            OnDevice d(k->dev);
            n += null_too && d.good && ws_give(P, i, nullptr);
        } else if (hipStream_t own = ws_own_stream(P, k->dev)) {
            n += ws_give(P, i, own);
        }
    }
    return n;
}

// The device's memory that no call holds, back with the device for an allocation for st that has
// failed. False: there was none.
bool ws_trim(int dev, hipStream_t st)
{
    WsPool &P = ws_pool();
    std::lock_guard<std::mutex> lock(P.mu);
    if (ws_give_all(P, dev, st == nullptr) == 0) return false;
    OnDevice d(dev);
    if (P.own[dev]) (void)ok(hipStreamSynchronize(P.own[dev]));
    if (!st) (void)ok(hipStreamSynchronize(nullptr));
    hipMemPool_t pool = nullptr;   // the runtime keeps freed memory until it is trimmed
    if (ok(hipDeviceGetDefaultMemPool(&pool, dev))) (void)ok(hipMemPoolTrimTo(pool, 0));
    return true;
}

// The device of st; false while st is being captured or where it cannot be told.
bool ws_device(hipStream_t st, int &dev)
{
    if (st) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        hipDevice_t sd = 0;
        if (!ok(hipStreamIsCapturing(st, &cap)) || cap != hipStreamCaptureStatusNone || !ok(hipStreamGetDevice(st, &sd)))
            return false;
        dev = (int)sd;
    } else if (!ok(hipGetDevice(&dev))) {
        return false;
    }
    return dev >= 0 && dev < WS_MAX_DEV;
}

// A kept block of at least `bytes` for a call on st, or nullptr: take a plain allocation.
WsBlock *ws_take(size_t bytes, hipStream_t st)
{
    WsPool &P = ws_pool();
    int dev = 0;
    const size_t size = ws_class(bytes);
    if (size > WS_KEEP_BYTES || !ws_device(st, dev)) return nullptr;
    std::lock_guard<std::mutex> lock(P.mu);
    if (P.handles <= 0) return nullptr;
    RelaxedCapture relaxed;
    WsBlock *best = nullptr;
    for (WsBlock *k : P.blocks) {
        if (k->busy || k->dev != dev || k->size < bytes || (best && best->size <= k->size)) continue;
        if (ws_ready(k, st)) best = k;
    }
    if (best && !ws_order(best, st)) best = nullptr;
    if (!best) {
        for (size_t i = P.blocks.size(); i-- > 0 && P.held[dev] + size > WS_KEEP_BYTES;) {
            const WsBlock *k = P.blocks[i];
            if (k->dev == dev && !k->busy && k->size < bytes && ws_ready(k, st)) (void)ws_give(P, i, st);
        }
        if (P.held[dev] + size > WS_KEEP_BYTES) return nullptr;
        void *p = nullptr;
        if (!ok(hipMallocAsync(&p, size, st))) return nullptr;
        best = new WsBlock{p, size, dev, st, nullptr, false, false};
        P.blocks.push_back(best);
        P.held[dev] += size;
    }
    best->busy = true;
    best->idle = false;
    best->last = st;
    return best;
}

}  // namespace

// After the call's last launch.
void ws_return(WsBlock *k, hipStream_t st)
{
    WsPool &P = ws_pool();
    std::lock_guard<std::mutex> lock(P.mu);
    RelaxedCapture relaxed;
    if (st) {
        const bool noted = (k->ev || ok(hipEventCreateWithFlags(&k->ev, hipEventDisableTiming))) && ok(hipEventRecord(k->ev, st));
        if (!noted) {   // no event: wait here, once; a block whose end is unknown is never lent again
            k->idle = ok(hipStreamSynchronize(st));
            if (!k->idle) return;
        }
    } else if (k->ev) {   // its next call is ordered by the null stream alone
        (void)ok(hipEventDestroy(k->ev));
        k->ev = nullptr;
    }
    k->busy = false;
    if (P.handles <= 0)
        for (size_t i = 0; i < P.blocks.size(); i++)
            if (P.blocks[i] == k) {
                (void)ws_give(P, i, st);
                break;
            }
}

void ws_handles(int d)
{
    WsPool &P = ws_pool();
    std::lock_guard<std::mutex> lock(P.mu);
    P.handles += d;
    if (P.handles <= 0) (void)ws_give_all(P, -1, true);
}

hipError_t scratch_alloc(StreamBuf &b, size_t bytes, hipStream_t st)
{
    b.st = st;
    if ((b.kept = ws_take(bytes, st))) {
        b.p = b.kept->p;
        return hipSuccess;
    }
    hipError_t e = hipMallocAsync(&b.p, bytes, st);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        int dev = 0;
        if (ws_device(st, dev) && ws_trim(dev, st) && (e = hipMallocAsync(&b.p, bytes, st)) != hipSuccess)
            (void)hipGetLastError();
    }
    if (e != hipSuccess) b.p = nullptr;
    return e;
}

hipError_t device_alloc(void **p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        int dev = 0;
        if (ws_device(nullptr, dev) && ws_trim(dev, nullptr) && (e = hipMalloc(p, bytes)) != hipSuccess)
            (void)hipGetLastError();
    }
    if (e != hipSuccess) *p = nullptr;
    return e;
}

}  // namespace k3kda
