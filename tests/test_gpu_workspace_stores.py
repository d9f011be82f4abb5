# SPDX-License-Identifier: Apache-2.0
"""Phase 1's two store policies (csrc/kda_chunk.hip): a pass whose workspace is above 200 MiB
stores it through to memory, a smaller one ordinarily. The same sequence in one pass above the
line and in passes below it gives the same bits, from fp32 and bf16 inputs and from prepared
ones (chunk boundaries do not move, and the policy only says where the bytes are kept)."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fp32", "bf16", "prepared"])
@pytest.mark.parametrize("D,H,T", [(128, 32, 2900), (64, 48, 5750)])
def test_store_policies_give_the_same_bits(gpu, D, H, T, form):
    import torch
    P, K, lb = H * D, 4, -5.0
    g = torch.Generator(device="cuda").manual_seed(T)
    rn = lambda *s: torch.randn(s, device="cuda", generator=g)
    assert gpu.kda_chunk_workspace(T, H, D) > 200 << 20 > gpu.kda_chunk_workspace(T // 2, H, D)
    q, k, v, z, b = rn(T, P), rn(T, P), rn(T, P), rn(T, P), rn(T, H)
    w = [rn(P, K) * 0.5 for _ in range(3)]
    A, dt, S0 = torch.rand(H, device="cuda", generator=g), rn(P), rn(H, D, D) * 0.1
    if form == "bf16":
        q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    if form == "prepared":
        q, k = (torch.nn.functional.normalize(t.view(T, H, D), dim=-1).view(T, P).contiguous() for t in (q, k))
        z, b = -5.0 * torch.sigmoid(z), torch.sigmoid(b)
    got = []
    for tokens in (T, T // 2):
        ws = torch.empty(gpu.kda_chunk_workspace(tokens, H, D), dtype=torch.uint8, device="cuda")
        S, hist, o = S0.clone(), torch.zeros(3, P, K - 1, device="cuda"), torch.empty(T, P, device="cuda")
        if form == "prepared":
            gpu.kda_chunk(q, k, v, z, b, S, o, H, D, D ** -0.5, workspace=ws)
        else:
            gpu.kda_prefill(q, k, v, z, b, *w, A, dt, hist, S, o, H, D, K, lb, D ** -0.5, ws)
        torch.cuda.synchronize()
        assert torch.isfinite(o).all()
        got.append((o, S, hist))
    for one, two in zip(*got):
        assert torch.equal(one, two)
