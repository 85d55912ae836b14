"""GPU: the MFMA GEMM (more than 16 rows) at the edges of its pipeline and tiles: K runs shorter than the pipeline is deep and with
every remainder of its unrolled loop, against the float64 oracle."""

import numpy as np
import pytest
import torch

from gpu_util import TORCH, assert_close, host_f64, logical_to_device, make_x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("kt", [1, 2, 3, 4, 5, 6, 7, 9, 11])
def test_short_k_runs(oracle, hm, device, dtype, kt):
    # kt K tiles of 128: fewer than the pipeline requests ahead, and each remainder behind its loop of whole trips. Several
    # calls on one output, so that activations of a K tile read too early would show as the previous call's or tile's.
    rng = np.random.default_rng(300 + kt)
    k, n, g = 128 * kt, 512, 128
    w_np = oracle.random_weights(rng, k, n, g, dtype)
    w = hm.RepackedMatrix.from_logical(*logical_to_device(w_np, dtype, device), g, dtype=TORCH[dtype])
    wf = oracle.weights_f64(*w_np, g, dtype)
    for m in (17, 64, 130):
        x64, x = make_x(oracle, rng, m, k, dtype, device)
        y = torch.full((m, n), float("nan"), dtype=TORCH[dtype], device=device)
        hm.packed_linear(y, x, w)
        y2 = torch.full_like(y, float("nan"))
        for _ in range(4):
            hm.packed_linear(y2, x, w)
        torch.cuda.synchronize()
        assert_close(oracle, host_f64(y), x64 @ wf, dtype, f"{kt} K tiles M={m}")
        assert torch.equal(y, y2)
