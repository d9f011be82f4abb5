# SPDX-License-Identifier: Apache-2.0
"""The MLA attention's head groups and head tiles (csrc/kda_mla_attn.hip) against the oracle at
the decode bar (rtol 1e-4, atol 1e-4 rms): head counts on both sides of each 16-head tile and
64-head group, groups of unequal size, contexts of one tile, several ranges and a ragged last
tile; and a latent wider than the one-pass kernel holds (the batched GEMM form, at a context for
each of its three softmax variants)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_close
from test_gpu_mla import mla_case, rms
import k3_oracle as ko

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,kvl,qr,B,start,gate", [
    (16, 512, 64, 2, 150, 1), (17, 64, 16, 3, 33, 0), (33, 512, 64, 1, 20, 1), (48, 64, 16, 25, 40, 1),
    (65, 512, 64, 2, 150, 1), (96, 512, 64, 3, 47, 1), (96, 32, 8, 17, 5, 0), (128, 64, 16, 2, 300, 1),
    (130, 48, 12, 1, 31, 1), (8, 528, 16, 2, 30, 1),
    (4, 528, 16, 1, 2100, 1), (4, 528, 16, 1, 8300, 1)])
def test_mla_head_groups_vs_oracle(gpu, H, kvl, qr, B, start, gate):
    """`start` cached positions written to both caches, then three steps."""
    import torch
    print(f"H={H} kv_lora={kvl} rope={qr} B={B} start={start} gate={gate}", flush=True)
    rng = np.random.default_rng(0x4B334441 + 0x60 + H + kvl + start)
    hidden, ql, qn, vh = 128, 32, 16, 16
    cfg, W = mla_case(rng, hidden, H, ql, kvl, qn, qr, vh, gate)
    cap = start + 5
    lat = rng.standard_normal((B, start, kvl)).astype(np.float32)
    rope = rng.standard_normal((B, start, qr)).astype(np.float32)
    up = (np.asarray(W.arrays["kv_b"], np.uint32) << 16).astype(np.uint32).view(np.float32).astype(np.float64)
    kvcs = [np.zeros((cap, H * (qn + vh)), np.float32) for _ in range(B)]
    ropecs = [np.zeros((cap, qr), np.float32) for _ in range(B)]
    for b in range(B):
        kvcs[b][:start] = lat[b].astype(np.float64) @ up.T
        ropecs[b][:start] = rope[b]
    cache = torch.zeros((B, cap, kvl + qr), device="cuda")
    cache[:, :start] = torch.from_numpy(np.concatenate([lat, rope], axis=2)).cuda()
    mw = gpu.MlaWeights(W.w, cfg)
    for t in range(start, start + 3):
        x = rng.standard_normal((B, hidden)).astype(np.float32)
        want = np.concatenate([ko.mla(x[b:b + 1], W, cfg, 1, kvcs[b], ropecs[b], t, cap) for b in range(B)])
        out = torch.full((B, hidden), float("nan"), device="cuda")
        mw.decode(out, torch.from_numpy(x).cuda(), cache, t, cap)
        torch.cuda.synchronize()
        r = assert_close(out.cpu().numpy(), want, 1e-4 * rms(want), 1e-4, f"H={H} position {t}")
        print(f"position {t}: {r:.3f}x", flush=True)
    mw.close()
