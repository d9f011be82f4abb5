# SPDX-License-Identifier: Apache-2.0
"""The products of csrc/kda_mid.hip where they can go wrong: one K-step, row counts around the 64-
and 128-row tiles, head counts whose q / k / v / gate blocks end inside a column tile, each tile
shape of both forms: bf16 rows (the prefill's z product) on 64 x 64, 64 x 128 and 128 x 128,
split fp32 rows (the full-accuracy layer) on 64 x 64 and 64 x 128; bf16 and fp32 inputs and
results. Held, like the other forms, to the oracle's k3_kda_layer: the bf16 prefill at
2e-3 (its bf16 results at twice that, the rounding of the result), the full-accuracy layer on
bf16 weights at 1e-4. The projected inputs in the conv history: the prefill's at 1e-5 (fp32 sums of
exact products), the split form's at 2^-17 sum |x| |w|, element by element (hi + lo leaves at most
2^-9 2^-9 |x| of each input; as much again for the fp32 sums).

The full-accuracy layer's S is held in the 2-norm, at 3e-5: the split products (hi + lo of each
operand, 2.5e-6 rms each, lo x lo left out, in the projections, the chunk factors and the state
update) put it 6e-6 to 8e-6 from 64 bits at these shapes, in any order of the sums. Element by
element against the rms of all heads that spread has no fixed bound: the rows of a head's slowly
decaying channels are many times the rms, and so are their errors (half a million elements at
32 x 128 heads)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_close
from test_gpu_layer_prefill import TOL, bf16_to_f32, layer_weights, rms
from test_oracle_ref import bf16
import k3_oracle as ko
from k3_oracle import f32

pytestmark = pytest.mark.gpu

SHAPES = [(64, 3, 64, (33, 64, 65)), (192, 5, 64, (127, 129)), (128, 2, 128, (40, 200)),
          (64, 32, 128, (63, 257)), (1024, 33, 64, (97,)), (64, 32, 128, (460, 900))]
CUS = 256


def tiles(hidden, H, D, T, dev):
    """The tile shapes of the layer's launches, by the kernel's rule (half the CUs' worth of
    256 x 256 tiles of z and more are not its own in the prefill)."""
    P = H * D
    wide = lambda rows: -(-rows // 128)
    if not dev:
        if 2 * -(-T // 256) * -(-P // 256) > CUS:
            return set()
        if wide(P) * -(-T // 128) >= CUS:
            return {(128, 128)}
        return {(64, 128) if wide(P) * -(-T // 64) >= CUS else (64, 64)}
    if T < 33:
        return set()
    return {(64, 128) if n * -(-T // 64) >= CUS else (64, 64) for n in (4 * wide(P) + wide(D + H), wide(P), wide(hidden))}


def test_every_tile_shape_is_reached():
    reached = lambda dev: set().union(*(tiles(h, H, D, T, dev) for h, H, D, Ts in SHAPES for T in Ts))
    assert reached(False) == {(64, 64), (64, 128), (128, 128)}
    assert reached(True) == {(64, 64), (64, 128)}


@pytest.mark.parametrize("dev", [False, True])
@pytest.mark.parametrize("hidden,H,D,Ts", SHAPES)
def test_short_prefill_projections_vs_oracle(gpu, hidden, H, D, Ts, dev):
    import torch
    rng = np.random.default_rng(0x4B334441 + 0x1D + hidden + H)
    K, P = 4, H * D
    W = layer_weights(rng, hidden, H, D, K)
    cfg = ko.make_cfg(hidden, H, D, K, -5.0, 1e-5)
    nst = P * D + 3 * P * (K - 1)
    st_ref = np.zeros(nst, np.float32)
    dw = gpu.DeviceWeights(W.w, cfg, gpu.UPLOAD_DEV if dev else gpu.UPLOAD_PREFILL)
    dst = torch.zeros(nst, device="cuda")
    for i, T in enumerate(Ts):
        x = f32(rng.standard_normal((T, hidden)))
        if not dev:
            x = bf16_to_f32(bf16(x))
        want = ko.kda_layer(ko.orc(), x, W, cfg, T, st_ref)
        dx = torch.from_numpy(x).cuda()
        half = not dev and i % 2 == 1                       # bf16 results
        out = torch.full((T, hidden), float("nan"), device="cuda", dtype=torch.bfloat16 if half else torch.float32)
        if dev:
            dw.layer(out, dx, dst, T)
        else:
            dw.layer_prefill(out, dx.to(torch.bfloat16) if (i + H) % 2 else dx, dst, T)
        torch.cuda.synchronize()
        tol = 1e-4 if dev else (2 * TOL if half else TOL)
        r = assert_close(out.float().cpu().numpy(), want, tol * rms(want), tol, f"T={T} out")
        got = dst.cpu().numpy()
        if dev:
            e = np.linalg.norm(np.float64(got[:P * D]) - st_ref[:P * D]) / np.linalg.norm(np.float64(st_ref[:P * D]))
            assert e <= 3e-5, f"T={T} S: {e:.2e} from the oracle"
        else:
            assert_close(got[:P * D], st_ref[:P * D], TOL * rms(st_ref[:P * D]), TOL, f"T={T} S")
        if dev:
            bound = np.stack([np.abs(x[1 - K:]).astype(np.float64) @ np.abs(bf16_to_f32(W.arrays[n])).T for n in ("q", "k", "v")])
            bound = 2.0 ** -17 * bound.transpose(0, 2, 1).ravel()     # [3][P][K - 1], as the history
            worst = float(np.max(np.abs(np.float64(got[P * D:]) - st_ref[P * D:]) / bound))
            assert worst <= 1.0, f"T={T} conv history: {worst:.3f}x the split's bound"
        else:
            assert_close(got[P * D:], st_ref[P * D:], 1e-5 * rms(st_ref[P * D:]), 1e-5, f"T={T} conv history")
        print(f"hidden={hidden} H={H} D={D} T={T} {'dev' if dev else 'prefill'}: worst {r:.3f}x", flush=True)
    dw.close()


def test_split_rows_and_tiles_give_the_same_bits(gpu):
    """The full-accuracy layer's longest prefills (at this width from 2e11 products of the input
    projections) run kda_mm.hip on 2T split rows and add the halves, shorter ones kda_mid.hip with
    an accumulator per half: a sequence in one call of the first kind and in two of the second
    (chunk boundaries do not move) is the same bits."""
    import torch
    hidden, H, D, K, T = 4096, 32, 128, 4, 3072
    P = H * D
    assert T / 2 * (4 * P + D + H) * hidden < 2e11 < T * (4 * P + D + H) * hidden and T // 2 % 64 == 0
    cfg = ko.make_cfg(hidden, H, D, K, -5.0, 1e-5)
    dw = gpu.DeviceWeights(layer_weights(np.random.default_rng(9), hidden, H, D, K).w, cfg, gpu.UPLOAD_DEV)
    x = torch.randn((T, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(9))
    got = []
    for n in (T, T // 2):
        st, out = torch.zeros(P * D + 3 * P * (K - 1), device="cuda"), torch.empty_like(x)
        for t in range(0, T, n):
            dw.layer(out[t:t + n], x[t:t + n], st, n)
        torch.cuda.synchronize()
        assert torch.isfinite(out).all()
        got.append((out, st))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    dw.close()
