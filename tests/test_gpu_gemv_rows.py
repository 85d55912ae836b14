"""GPU: five to sixteen rows at the edges of the launch rules: projections narrow enough for one unsplit launch of strip pairs or
single strips, on both sides of one and two strips per CU and of the K it takes, and K that does not fit the workgroup's memory
whole and is split, against the float64 oracle."""

import numpy as np
import pytest
import torch

from gpu_util import TORCH, assert_close, host_f64, logical_to_device, make_x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("k,n,group", [
    (128, 16, 32), (384, 48, 64), (1024, 4096, 128), (3968, 4112, 128), (4096, 4096, 64), (4096, 1040, 32), (2688, 8192, 64),
    (2688, 8208, 128), (5120, 2064, 64), (5248, 512, 32), (8192, 256, 64), (14336, 1024, 128), (2048, 1024, 64), (2176, 528, 32),
    (3968, 6144, 32), (4608, 2560, 128), (4608, 1024, 64), (7680, 1024, 64)])
def test_rows(oracle, hm, device, k, n, group, dtype):
    # 16 to 8208 columns: 1, odd counts, 256, 257, 512 and 513 strips; 1, 3, 8, 31, 32, 40, 41, 64 and 112 K tiles; in groups of 32
    # and 64 eight waves of 16, 17 and 31 K tiles; 36 and 60 K tiles with enough strips to run unsplit and with too few. The
    # frame around the output has to stay untouched.
    rng = np.random.default_rng(360 + k + n)
    w_np = oracle.random_weights(rng, k, n, group, dtype)
    w = hm.RepackedMatrix.from_logical(*logical_to_device(w_np, dtype, device), group, dtype=TORCH[dtype])
    wf = oracle.weights_f64(*w_np, group, dtype)
    for m in (5, 8, 9, 12, 13, 16):
        x64, x = make_x(oracle, rng, m, k, dtype, device)
        frame = torch.full((m + 2, n + 32), 7.0, dtype=TORCH[dtype], device=device)
        y = frame[1:m + 1, 16:n + 16]
        hm.packed_linear(y, x, w)
        y2 = torch.empty((m, n), dtype=TORCH[dtype], device=device)
        hm.packed_linear(y2, x, w)
        torch.cuda.synchronize()
        assert_close(oracle, host_f64(y), x64 @ wf, dtype, f"linear {k}x{n} g={group} M={m}")
        assert torch.equal(y, y2), (k, n, m)
        frame[1:m + 1, 16:n + 16] = 7.0
        assert bool((frame == 7.0).all()), (k, n, m)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("hidden,inter,group", [(256, 128, 128), (2048, 512, 64), (4096, 1024, 32), (5120, 4096, 128)])
def test_rows_fused(oracle, hm, device, hidden, inter, group, dtype):
    # The fused gate_up unsplit (8 to 256 strip pairs) or, in groups of 32, split, and the down behind it.
    rng = np.random.default_rng(370 + hidden)
    ws = [oracle.random_weights(rng, hidden, inter, group, dtype), oracle.random_weights(rng, hidden, inter, group, dtype),
          oracle.random_weights(rng, inter, hidden, group, dtype)]
    layer = hm.FfnLayer.from_logical(*(logical_to_device(t, dtype, device) for t in ws), group, dtype=TORCH[dtype])
    wg, wu = (oracle.weights_f64(*t, group, dtype) for t in ws[:2])
    for m in (5, 9, 16):
        x64, x = make_x(oracle, rng, m, hidden, dtype, device)
        act = layer.gate_up(x)
        torch.cuda.synchronize()
        g = x64 @ wg
        assert_close(oracle, host_f64(act), g / (1 + np.exp(-g)) * (x64 @ wu), dtype, f"gate_up {hidden}x{inter} M={m}")
