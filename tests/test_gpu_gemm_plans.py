"""GPU: every instantiation of the prefill GEMM (tile shape, group, type, plain and fused) at the lengths of its K runs where its
pipeline takes another path, on the launches listed in gemm_cases.py.

Plain calls use integer activations and scales that are powers of two: every product and every partial sum is then exact in fp32
(multiples of 2^-7 below 2^14) in any order of summation, so the output has to be the exact result's rounding, bit for bit."""

import pytest
import torch

from gemm_cases import TILES, gemm_plan
from gpu_util import TORCH, assert_close, host_f64

pytestmark = pytest.mark.gpu


def _logical(gen, k, n, group, dtype, scales):
    q = torch.randint(0, 16, (k, n), dtype=torch.uint8, device="cuda", generator=gen)
    z = torch.randint(0, 17, (k // group, n), dtype=torch.uint8, device="cuda", generator=gen)
    return q, scales((k // group, n)).to(TORCH[dtype]), z


def _dense(q, s, z, group):
    """(q - z) s in float64."""
    k, n = q.shape
    w = (q.view(k // group, group, n).double() - z.view(k // group, 1, n).double()) * s.view(k // group, 1, n).double()
    return w.view(k, n)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("tile", sorted(TILES))
def test_plain_exact(hm, device, tile, group, dtype):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(390 + tile)
    cases = TILES[tile]
    k_max, n_max = 128 * max(c[2] for c in cases), max(c[1] for c in cases)
    mat = _logical(gen, k_max, n_max, group, dtype, lambda shape: torch.exp2(torch.randint(-7, -3, shape, device="cuda", generator=gen).float()))
    w = hm.RepackedMatrix.from_logical(*mat, group, dtype=TORCH[dtype])
    for m, cols, kt, splits in cases:
        k = 128 * kt
        plan = gemm_plan(m, cols, k)
        assert (plan.tile, plan.splits) == (tile, splits)
        x = torch.randint(-2, 3, (m, k), device="cuda", generator=gen).to(TORCH[dtype])
        exact = x.double() @ _dense(mat[0][:k, :cols], mat[1][:k // group, :cols], mat[2][:k // group, :cols], group)
        ref = exact.to(TORCH[dtype])
        frame = torch.full((m + 1, cols + 16), 7.0, dtype=TORCH[dtype], device=device)
        y = frame[:m, :cols]
        hm.packed_linear(y, x, w, k=k, n=cols)
        pair = torch.full((m, cols), float("nan"), dtype=TORCH[dtype], device=device)
        hm.packed_linear_k_split(pair, torch.cat([x, x], dim=1), w, w, k0=k, k1=k, n=cols)  # the second share adds into the output
        torch.cuda.synchronize()
        print(f"tile {tile} g={group} {dtype} M={m} N={cols} K={k} splits={splits}", flush=True)
        assert torch.equal(y, ref), (m, cols, kt, int((y != ref).sum()))
        assert torch.equal(pair, ref + ref), (m, cols, kt)
        y.fill_(7.0)
        assert bool((frame == 7.0).all()), (m, cols, kt)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("tile", sorted(TILES))
def test_fused(oracle, hm, device, tile, group, dtype):
    # One unsplit call and the K splits of the tile (SwiGLU after the K groups' exchange, and in the split sum). Layers have
    # channels in multiples of 128.
    gen = torch.Generator(device="cuda")
    gen.manual_seed(391 + tile)
    fit = [c for c in TILES[tile] if c[1] % 256 == 0]
    cases = [c for c in fit if c[3] == 1][1:2] or [c for c in fit if c[3] == 1]
    cases += [c for c in fit if c[3] > 1]
    assert cases and cases[0][3] == 1 and cases[-1][3] > 1
    for m, cols, kt, splits in cases:
        h, i = 128 * kt, cols // 2
        plan = gemm_plan(m, cols, h)
        assert (plan.tile, plan.splits) == (tile, splits)
        mats = [_logical(gen, *s, group, dtype, lambda shape: torch.rand(shape, device="cuda", generator=gen) * 0.019 + 0.001)
                for s in ((h, i), (h, i), (i, h))]
        layer = hm.FfnLayer.from_logical(*mats, group, dtype=TORCH[dtype])
        x = (torch.randn((m, h), device="cuda", generator=gen) / 8).to(TORCH[dtype])
        act = layer.gate_up(x)
        torch.cuda.synchronize()
        gate, up = (x.double() @ _dense(*t, group) for t in mats[:2])
        ref = gate / (1 + torch.exp(-gate)) * up
        assert_close(oracle, host_f64(act), ref.cpu().numpy(), dtype, f"tile {tile} g={group} gate_up {h}x{i} M={m} splits={splits}")
