"""GPU: calls with an explicit stream that is not torch's current one. What a call allocates for itself (split partials, a layer's
workspace, results it returns) belongs to that stream: a block of the current stream's pool could still be in use there, and would
go back to it while the call's kernels run."""

import numpy as np
import pytest
import torch

import heteromega_amd.ffn as ffn
from gpu_util import TORCH, assert_close, host_f64, logical_to_device, make_x

pytestmark = pytest.mark.gpu


class _Allocations:
    """torch.empty and torch.zeros as heteromega_amd sees them, noting the stream each device tensor is made on."""

    def __init__(self, monkeypatch):
        self.streams = []
        for name in ("empty", "zeros"):
            monkeypatch.setattr(torch, name, self._noting(getattr(torch, name)))

    def _noting(self, fn):
        def made(*args, **kwargs):
            t = fn(*args, **kwargs)
            if t.is_cuda:
                self.streams.append(torch.cuda.current_stream().cuda_stream)
            return t
        return made


def _matrix(oracle, hm, rng, k, n, dtype, device):
    w = oracle.random_weights(rng, k, n, 128, dtype)
    return oracle.weights_f64(*w, 128, dtype), hm.RepackedMatrix.from_logical(*logical_to_device(w, dtype, device), 128, dtype=TORCH[dtype])


@pytest.mark.parametrize("kind", ["torch", "handle", "external"])
def test_allocations_on_the_calls_stream(oracle, hm, device, monkeypatch, kind):
    rng = np.random.default_rng(380)
    dtype, k, n, m = "fp16", 4096, 512, 100  # a GEMM that divides its K range
    wf, w = _matrix(oracle, hm, rng, k, n, dtype, device)
    x64, x = make_x(oracle, rng, m, k, dtype, device)
    mats = [oracle.random_weights(rng, *s, 128, dtype) for s in ((1024, 1024), (1024, 1024), (1024, 1024))]
    layer = hm.FfnLayer.from_logical(*(logical_to_device(t, dtype, device) for t in mats), 128, dtype=TORCH[dtype])
    _, xf = make_x(oracle, rng, m, 1024, dtype, device)
    norm = torch.ones(1024, dtype=TORCH[dtype], device=device)
    assert w.workspace_bytes(m) > 0
    out = torch.zeros((m, n), dtype=TORCH[dtype], device=device)
    out2 = torch.zeros((m, n), dtype=TORCH[dtype], device=device)
    x2 = torch.cat([x, x], dim=1)
    s = torch.cuda.Stream()
    stream = {"torch": s, "handle": s.cuda_stream, "external": torch.cuda.ExternalStream(s.cuda_stream)}[kind]
    plain = layer.forward(xf[:40])
    torch.cuda.synchronize()
    seen = _Allocations(monkeypatch)
    ffn.packed_linear(out, x, w, stream=stream)
    ffn.packed_linear_k_split(out2, x2, w, w, stream=stream)
    hm.hetero.hetero_linear(out, x, None, w, stream=stream)
    y = layer.forward(xf[:40], stream=stream)
    layer.forward(xf, stream=stream)  # the layer's workspace grows
    layer.down(layer.gate_up(xf, stream=stream), stream=stream)
    layer.block_forward(xf.clone(), norm, stream=stream)
    reduced, _ = ffn.ffn_partitioned(layer, xf[:40], ffn.FFNPartition(1024, 0), stream=stream)
    w.dequantize(stream=stream)
    w.to_logical(stream=stream)
    assert ffn.find_nonfinite(xf, stream=stream) == -1
    assert len(seen.streams) >= 12 and set(seen.streams) == {s.cuda_stream}
    monkeypatch.undo()
    torch.cuda.synchronize()
    assert_close(oracle, host_f64(out), x64 @ wf, dtype, "packed_linear on another stream")
    assert torch.equal(out2, out + out)
    assert torch.equal(y, plain) and torch.equal(reduced, plain)


def test_current_stream_reuses_nothing_in_flight(oracle, hm, device):
    # The call waits behind a long kernel on its stream while the current stream allocates and writes blocks of the sizes that
    # the call uses.
    rng = np.random.default_rng(381)
    dtype, k, n, m = "bf16", 4096, 512, 100
    wf, w = _matrix(oracle, hm, rng, k, n, dtype, device)
    x64, x = make_x(oracle, rng, m, k, dtype, device)
    need = w.workspace_bytes(m) + 256
    s = torch.cuda.Stream()
    out = torch.empty((m, n), dtype=TORCH[dtype], device=device)
    for i in range(3):
        out.fill_(float("nan"))
        held = [torch.full((need,), 0xFF, dtype=torch.uint8, device=device) for _ in range(4)]
        del held  # blocks of the current stream's pool, free again
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            torch.cuda._sleep(50_000_000)
        ffn.packed_linear(out, x, w, stream=s)
        held = [torch.full((need,), 0xFF, dtype=torch.uint8, device=device) for _ in range(8)]
        torch.cuda.synchronize()
        assert_close(oracle, host_f64(out), x64 @ wf, dtype, f"packed_linear behind a busy stream, call {i}")
        del held
