# SPDX-License-Identifier: Apache-2.0
"""The double-accumulating projections of k3hip_kda_layer_dev (csrc/kda_proj.hip) at the edges
of their forms: token counts around the GEMV / MFMA switch (4 | 5) and the 16-token tiles,
hidden widths below, at and past one 512-wide block with and without whole 8-element slices,
row counts on both sides of the one / two rows a wave rule (8192), two rows a wave over one block,
over five and over seven (four at a time, then two, then the last with one slice), each weight
format.

The layer's conv history holds the last K - 1 projected q, k, v: double sums rounded once to
fp32 (int8: the double sum of the int8 products rounded to fp32, times the row's fp32 scale).
They are compared with the same sums by numpy in float64, whose other order moves the double
sum by far less than 1e-9 for at most 3080 products of order one: at most one unit in the last
place, 2^-23 relative (two for int8, whose product with the scale rounds once more). Output and
state are held to the oracle's k3_kda_layer at the layer's 1e-4 bar.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_close
from test_gpu_dropin import q8_layer
from test_gpu_layer_prefill import bf16_to_f32, layer_weights, rms
import k3_oracle as ko
from k3_oracle import f32

pytestmark = pytest.mark.gpu


def project(w, wdt, hidden, x):
    """x . w^T in float64, rounded as the format's GEMV rounds it."""
    if wdt == "int8":
        rows = np.ascontiguousarray(w).view(np.uint8).reshape(-1, 4 + hidden)
        scale = np.ascontiguousarray(rows[:, :4]).view(np.float32)[:, 0]
        return (x.astype(np.float64) @ rows[:, 4:].view(np.int8).astype(np.float64).T).astype(np.float32) * scale
    w = bf16_to_f32(w) if wdt == "bf16" else w
    return (x.astype(np.float64) @ w.astype(np.float64).T).astype(np.float32)


@pytest.mark.parametrize("wdt", ["fp32", "bf16", "int8"])
@pytest.mark.parametrize("hidden,H,D,Ts", [(72, 3, 64, (1, 2, 3, 4, 5, 16, 17, 32, 33, 70)),
                                           (100, 2, 64, (1, 3, 5, 20)), (1104, 1, 128, (4, 1, 15, 49, 65)),
                                           (136, 16, 128, (1, 2, 4)), (2056, 16, 128, (1, 2, 3)),
                                           (3080, 16, 128, (1, 2, 4))])
def test_projection_forms_vs_oracle(gpu, hidden, H, D, Ts, wdt):
    import torch
    rng = np.random.default_rng(0x4B334441 + 0x90 + hidden + D)
    K, P = 4, H * D
    if wdt == "int8":
        W = q8_layer(rng, hidden, H, D, K)
    else:
        W = layer_weights(rng, hidden, H, D, K)
        if wdt == "fp32":
            W = ko.Weights({n: (bf16_to_f32(a) if a.dtype == np.uint16 else a) for n, a in W.arrays.items()}, 0)
    cfg = ko.make_cfg(hidden, H, D, K, -5.0, 1e-5)
    nst = P * D + 3 * P * (K - 1)
    st_ref = np.zeros(nst, np.float32)
    dw = gpu.DeviceWeights(W.w, cfg, gpu.UPLOAD_DEV)
    dst = torch.zeros(nst, device="cuda")
    seen = np.zeros((K - 1, hidden), np.float32)   # the newest inputs; zeros before the first
    for T in Ts:
        print(f"hidden={hidden} H={H} D={D} {wdt} T={T}", flush=True)
        x = f32(rng.standard_normal((T, hidden)))
        want = ko.kda_layer(ko.orc(), x, W, cfg, T, st_ref)
        out = torch.full((T, hidden), float("nan"), device="cuda")
        dw.layer(out, torch.from_numpy(x).cuda(), dst, T)
        torch.cuda.synchronize()
        got = dst.cpu().numpy()
        seen = np.concatenate([seen, x])[-(K - 1):]
        hist = np.stack([project(W.arrays[n], wdt, hidden, seen).T for n in ("q", "k", "v")])
        assert_close(got[P * D:], hist, 1e-9, 2.0 ** (-22 if wdt == "int8" else -23), f"T={T} projections")
        assert_close(got[:P * D], st_ref[:P * D], 1e-4 * rms(st_ref[:P * D]), 1e-4, f"T={T} S")
        assert_close(out.cpu().numpy(), want, 1e-4 * rms(want), 1e-4, f"T={T} out")
    # one token of a fresh sequence (no state)
    x = f32(rng.standard_normal((1, hidden)))
    want = ko.kda_layer(ko.orc(), x, W, cfg, 1, None)
    out = torch.full((1, hidden), float("nan"), device="cuda")
    dw.layer(out, torch.from_numpy(x).cuda(), None, 1)
    torch.cuda.synchronize()
    assert_close(out.cpu().numpy(), want, 1e-4 * rms(want), 1e-4, "one token without a state")
    dw.close()
