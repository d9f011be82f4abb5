# SPDX-License-Identifier: Apache-2.0
"""Layer calls captured into a graph take scratch of the graph's own, not the kept blocks: each
replay gives the eager bits, with eager calls of the same weights (which use the kept blocks) and
synchronisations between the replays. And a capture that is open on one stream, in its global mode,
leaves eager calls on another stream, with blocks to look up there, what they are."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_layer_prefill import layer_weights
from test_gpu_mla import mla_case
import k3_oracle as ko

pytestmark = pytest.mark.gpu

HIDDEN, H, D, K = 512, 4, 128, 4
NST = H * D * D + 3 * H * D * (K - 1)


def _layer(gpu, kind):
    """(run(out, state, stream), out shape, state, close) of one kind of call; state is updated in place."""
    import torch
    rng = np.random.default_rng(0x4B334441 + 0x6C)
    g = torch.Generator(device="cuda").manual_seed(3)
    rn = lambda *s: torch.randn(s, device="cuda", generator=g)
    if kind == "mla":
        cfg, W = mla_case(rng, 256, 24, 64, 512, 32, 64, 32, 1)
        mw, x = gpu.MlaWeights(W.w, cfg), rn(3, 256)
        return (lambda out, st, stream=None: mw.decode(out, x, st, 70, 71, stream=stream)), (3, 256), rn(3, 71, 576), mw.close
    dw = gpu.DeviceWeights(layer_weights(rng, HIDDEN, H, D, K).w, ko.make_cfg(HIDDEN, H, D, K, -5.0, 1e-5))
    n = {"decode": 5, "token": 1, "short": 20, "long": 100}[kind]
    x = rn(n, HIDDEN)
    if kind == "decode":
        return (lambda out, st, stream=None: dw.layer_decode(out, x, st, NST, stream=stream)), (n, HIDDEN), 0.1 * rn(n, NST), dw.close
    return (lambda out, st, stream=None: dw.layer(out, x, st, n, stream=stream)), (n, HIDDEN), 0.1 * rn(NST), dw.close


@pytest.mark.parametrize("kind", ["decode", "token", "short", "long", "mla"])
def test_captured_calls_replay_the_eager_bits(gpu, kind):
    import torch
    print(kind, flush=True)
    run, shape, state0, close = _layer(gpu, kind)
    want, st = [], state0.clone()
    for _ in range(4):
        out = torch.full(shape, float("nan"), device="cuda")
        run(out, st)
        torch.cuda.synchronize()
        want.append((out, st.clone()))
    st, out = state0.clone(), torch.empty(shape, device="cuda")
    side = torch.cuda.Stream()
    eager_st, eager_out = state0.clone(), torch.empty(shape, device="cuda")
    with torch.cuda.stream(side):
        run(eager_out, eager_st, side)                # the side stream has a kept block, with its event
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="global"):
        run(out, st)
        run(eager_out, eager_st, side)                # eager, beside the open capture
    torch.cuda.synchronize()
    assert torch.equal(eager_out, want[1][0]) and torch.equal(eager_st, want[1][1])
    assert torch.equal(st, state0)                    # captured, not run
    other, other_out = state0.clone(), torch.empty(shape, device="cuda")
    for w_out, w_st in want:
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, w_out) and torch.equal(st, w_st)
        run(other_out, other)
        torch.cuda.synchronize()
        assert torch.equal(other_out, w_out) and torch.equal(other, w_st)
    del graph
    close()
