// SPDX-License-Identifier: Apache-2.0
// kda_scratch.h - device scratch of one call: a block kept between calls or a stream allocation
// (kda_scratch.hip).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>

namespace k3kda {

struct WsBlock;
void ws_return(WsBlock *k, hipStream_t st);
// A weight set was uploaded (+1) or released (-1); blocks are kept only while any is there.
void ws_handles(int d);

// Given back in stream order when the StreamBuf goes.
struct StreamBuf {
    void *p = nullptr;
    hipStream_t st = nullptr;
    WsBlock *kept = nullptr;
    ~StreamBuf()
    {
        if (kept) ws_return(kept, st);
        else if (p) (void)hipFreeAsync(p, st);
    }
};

// b.p = at least `bytes` of device memory for work on st.
hipError_t scratch_alloc(StreamBuf &b, size_t bytes, hipStream_t st);
// hipMalloc for what outlives a call (weights, states).
hipError_t device_alloc(void **p, size_t bytes);

}  // namespace k3kda
