# SPDX-License-Identifier: Apache-2.0
"""The two forms of the MLA decode attention over head counts, against the oracle at the decode
bar (rtol 1e-4, atol 1e-4 rms): up to 64 heads the one-pass kernel (csrc/kda_mla_attn.hip), on both
sides of each 16-head tile, over contexts of one tile, several ranges and a ragged last tile; more
heads, or a latent wider than that kernel holds, the batched fp32 GEMMs, at a context for each of
their three softmax variants. And the accuracy of more than 64 heads, whose attention works on all
24 bits, against 64 bits with the scores of small and of larger spread."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_close
from test_gpu_mla import mla_case, rms
from test_oracle_ref import bf16
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


@pytest.mark.parametrize("H,std", [(65, 1.0), (96, 1.0), (96, 5.0)])
def test_mla_beyond_64_heads_keeps_fp32_scores(gpu, H, std):
    """The layer's error against 64 bits, for scores of spread `std`. A score is a sum of 576 fp32
    products; its roundings, at most 2^-24 of it each, add up like a random walk, and its error is
    the relative error of its weight: 2^-24 sqrt(576) std. (Operands on 16 bits leave 3.5e-6 std,
    two and a half times that.) The layer's other products add 4e-7."""
    import torch
    rng = np.random.default_rng(0x4B334441 + 0x77 + H + int(10 * std))
    hidden, ql, kvl, qn, qr, vh, B, n = 256, 64, 512, 16, 64, 16, 2, 1000
    cfg, W = mla_case(rng, hidden, H, ql, kvl, qn, qr, vh, 1)
    QH = qn + qr
    c = std * np.sqrt(QH / (0.25 * qn + qr))               # rms of q for that spread
    arrays = dict(W.arrays, q_b=bf16(rng.standard_normal((H * QH, ql)) * (c / np.sqrt(ql))))
    W = ko.MlaWeights(arrays, 1)
    m = {k: (np.asarray(a, np.uint32) << 16).view(np.float32).astype(np.float64) if a.dtype == np.uint16
         else a.astype(np.float64) for k, a in arrays.items()}
    cache = rng.standard_normal((B, n + 1, kvl + qr)).astype(np.float32)
    x = rng.standard_normal((B, hidden)).astype(np.float32)

    norm = lambda v, w: v / np.sqrt((v * v).mean(-1, keepdims=True) + 1e-5) * w
    x64, c64 = x.astype(np.float64), cache.astype(np.float64)
    kv = x64 @ m["kv_a"].T
    c64[:, n] = np.concatenate([norm(kv[:, :kvl], m["kv_a_norm"]), kv[:, kvl:]], axis=1)
    q = (norm(x64 @ m["q_a"].T, m["q_a_norm"]) @ m["q_b"].T).reshape(B, H, QH)
    up = m["kv_b"].reshape(H, qn + vh, kvl)
    qc = np.concatenate([np.einsum("bhk,hkc->bhc", q[..., :qn], up[:, :qn]), q[..., qn:]], axis=2)
    s = np.einsum("bhc,bnc->bhn", qc, c64) / np.sqrt(QH)
    assert 0.8 * std < s.std() < 1.25 * std
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    o = np.einsum("bhn,bnc->bhc", p, c64[..., :kvl])
    o = np.einsum("bhc,hvc->bhv", o, up[:, qn:]).reshape(B, H * vh)
    want = (o / (1 + np.exp(-(x64 @ m["g"].T)))) @ m["o"].T

    mw = gpu.MlaWeights(W.w, cfg)
    out = torch.full((B, hidden), float("nan"), device="cuda")
    mw.decode(out, torch.from_numpy(x).cuda(), torch.from_numpy(cache).cuda(), n, n + 1)
    torch.cuda.synchronize()
    e = np.linalg.norm(out.cpu().numpy() - want) / np.linalg.norm(want)
    bar = 2.0 ** -24 * np.sqrt(576) * std + 4e-7
    print(f"H={H} std={std}: {e:.2e} from 64 bits, bar {bar:.2e}", flush=True)
    mw.close()
    assert e <= bar
