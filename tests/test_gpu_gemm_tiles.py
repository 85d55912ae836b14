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


@pytest.mark.parametrize("group", [32, 64, 128])
def test_bf16_weights_are_rounded_once(oracle, hm, device, group):
    # The rows of the identity through the GEMM give back the weights it multiplied with: bf16((q - z) s), rounded once from
    # the exact product, for every nibble position and value, zero points 0..16 and scales over 2^-100 .. 2^100.
    rng = np.random.default_rng(310 + group)
    k, n = 256, 512
    q = rng.integers(0, 16, (k, n), dtype=np.uint8)
    z = rng.integers(0, 17, (k // group, n), dtype=np.uint8)
    s = oracle.to_bits((rng.uniform(1, 2, (k // group, n)) * np.exp2(rng.integers(-100, 101, (k // group, n)))).astype(np.float32), "bf16")
    w = hm.RepackedMatrix.from_logical(*logical_to_device((q, s, z), "bf16", device), group, dtype=torch.bfloat16)
    x = torch.eye(k, dtype=torch.bfloat16, device=device)
    y = torch.empty((k, n), dtype=torch.bfloat16, device=device)
    hm.packed_linear(y, x, w)
    torch.cuda.synchronize()
    exact = (q.astype(np.float64) - np.repeat(z, group, 0)) * np.repeat(oracle.from_bits(s, "bf16").astype(np.float64), group, 0)
    np.testing.assert_array_equal(host_f64(y), oracle.from_bits(oracle.to_bits(exact.astype(np.float32), "bf16"), "bf16").astype(np.float64))
