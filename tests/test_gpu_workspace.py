# SPDX-License-Identifier: Apache-2.0
"""The scratch kept between calls: calls in flight on several streams and from several threads
never share a block, blocks of a finished stream are taken up by another one, and small and
large calls may alternate. Every result is compared bit for bit with the same call made alone
(all entry points used here are deterministic)."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from test_gpu_layer_prefill import layer_weights
import k3_oracle as ko

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads", [0, 3])
def test_workspaces_of_calls_in_flight(gpu, threads):
    import torch
    hidden, H, D, K = 512, 4, 128, 4
    P = H * D
    n = P * D + 3 * P * (K - 1)
    rng = np.random.default_rng(0x4B334441 + 77)
    cfg = ko.make_cfg(hidden, H, D, K, -5.0, 1e-5)
    dw = gpu.DeviceWeights(layer_weights(rng, hidden, H, D, K).w, cfg)
    g = torch.Generator(device="cuda").manual_seed(5)
    lens = (1, 70, 1500, 3, 400, 64)
    xs = [torch.randn((T, hidden), device="cuda", generator=g) for T in lens]

    def call(i, st, stream):
        out = torch.empty_like(xs[i])
        with torch.cuda.stream(stream):
            st.zero_()
            (dw.layer if i % 2 else dw.layer_prefill)(out, xs[i], st, lens[i], stream=stream)
        return out

    cur = torch.cuda.current_stream()
    states = [torch.empty(n, device="cuda") for _ in lens]
    want = []
    for i in range(len(lens)):
        o = call(i, states[i], cur)
        torch.cuda.synchronize()
        want.append((o, states[i].clone()))

    def rounds(k):
        try:
            compared.append(_rounds(k))
        except BaseException as e:          # an exception would end in the thread: it fails the test here
            bad.append((k, repr(e)))

    def _rounds(k):
        done = 0
        own = [torch.empty(n, device="cuda") for _ in lens]
        for r in range(3):
            streams = [torch.cuda.Stream(), torch.cuda.Stream()] + ([] if k else [cur])
            outs = [call(i, own[i], streams[(i + r) % len(streams)]) for i in range(len(lens))]
            for s in streams:
                s.synchronize()
            for i in range(len(lens)):
                if not (torch.equal(outs[i], want[i][0]) and torch.equal(own[i], want[i][1])):
                    bad.append((k, r, i))
                done += 1
        return done

    bad: list = []
    compared: list = []
    torch.cuda.synchronize()
    if threads:
        ts = [threading.Thread(target=rounds, args=(k + 1,)) for k in range(threads)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    else:
        rounds(0)
    dw.close()
    assert not bad, bad
    assert compared == [3 * len(lens)] * max(threads, 1)
