# SPDX-License-Identifier: Apache-2.0
"""k3hip_set_projection_gemm means what it says at every length: with K3HIP_GEMM_HIPBLASLT (the
default) the 4096-deep projections of a layer prefill (q / k / v, f_a with b, gate, o_proj) are
hipBLASLt's, short prompts among them, with K3HIP_GEMM_HANDWRITTEN none is; read from the names of
the kernels that a call launched."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_layer_prefill import layer_weights
import k3_oracle as ko

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [16, 333, 2500])
def test_the_setting_names_the_kernels(gpu, T):
    import torch
    from torch.profiler import ProfilerActivity, profile
    hidden, H, D, K = 512, 4, 128, 4
    cfg = ko.make_cfg(hidden, H, D, K, -5.0, 1e-5)
    dw = gpu.DeviceWeights(layer_weights(np.random.default_rng(3), hidden, H, D, K).w, cfg, gpu.UPLOAD_PREFILL)
    x = torch.randn((T, hidden), device="cuda").to(torch.bfloat16)
    out = torch.empty((T, hidden), device="cuda")
    names = {}
    for impl in (gpu.GEMM_HIPBLASLT, gpu.GEMM_HANDWRITTEN):
        gpu.set_projection_gemm(impl)
        try:
            dw.layer_prefill(out, x, None, T)
            torch.cuda.synchronize()
            with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
                dw.layer_prefill(out, x, None, T)
                torch.cuda.synchronize()
        finally:
            gpu.set_projection_gemm(gpu.GEMM_HIPBLASLT)
        names[impl] = [e.name for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA]
        print(f"T={T} setting {impl}:", *(n[:60] for n in names[impl]), sep="\n  ", flush=True)
    library = {i: sum(n.startswith("Cijk_") for n in ns) for i, ns in names.items()}
    assert any("kda_chunk_state" in n for n in names[gpu.GEMM_HIPBLASLT])     # the call's kernels are seen
    assert library == {gpu.GEMM_HIPBLASLT: 4, gpu.GEMM_HANDWRITTEN: 0}
    dw.close()
