"""GPU: the MFMA GEMM (more than 16 rows) at short K runs, at bf16 scales of any size, and at row counts on both sides of 32 to 128
rows on narrow matrices, against the float64 oracle. Every tile shape at every length of its K runs: test_gpu_gemm_plans.py."""

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


def _any_scales(rng, oracle, shape, lo, hi):
    bits = oracle.to_bits((rng.uniform(1, 1.99, shape) * np.exp2(rng.integers(lo, hi, shape))).astype(np.float32), "bf16")
    return bits, oracle.from_bits(bits, "bf16").astype(np.float64)


@pytest.mark.parametrize("group", [32, 64, 128])
def test_bf16_scales_of_any_size(oracle, hm, device, group):
    # The weights that the GEMM multiplies with, read back by the rows of the identity, over every bf16 scale: subnormal ones
    # (from 2^-133) to the largest, where (1024 + z) s leaves fp32 long before the weight leaves bf16. A weight beyond bf16 is
    # infinite. Also in a matrix joined from one without large scales and one with, and with K splits.
    rng = np.random.default_rng(320 + group)
    k, n = 256, 512
    x = torch.eye(k, dtype=torch.bfloat16, device=device)
    parts, exact = [], []
    for lo, hi in ((-133, 117), (-133, 128), (116, 128)):
        q = rng.integers(0, 16, (k, n), dtype=np.uint8)
        z = rng.integers(0, 17, (k // group, n), dtype=np.uint8)
        bits, s = _any_scales(rng, oracle, (k // group, n), lo, hi)
        w = hm.RepackedMatrix.from_logical(*logical_to_device((q, bits, z), "bf16", device), group, dtype=torch.bfloat16)
        with np.errstate(over="ignore"):
            e = ((q.astype(np.float64) - np.repeat(z, group, 0)) * np.repeat(s, group, 0)).astype(np.float32)
            e = torch.from_numpy(e).to(torch.bfloat16)
        # one row's product with an infinite weight of another row is 0 * inf: only columns of finite weights come back
        fine = torch.isfinite(e).all(dim=0)
        assert bool(fine.any())
        y = torch.empty((k, n), dtype=torch.bfloat16, device=device)
        hm.packed_linear(y, x, w)
        torch.cuda.synchronize()
        assert torch.equal(y.cpu()[:, fine], e[:, fine]), (lo, hi)
        parts.append(w)
        exact.append((e, fine))
    joined = hm.RepackedMatrix.concat(parts[:2])
    y = torch.empty((k, 2 * n), dtype=torch.bfloat16, device=device)
    hm.packed_linear(y, x, joined)
    torch.cuda.synchronize()
    for i, (e, fine) in enumerate(exact[:2]):
        assert torch.equal(y.cpu()[:, i * n:(i + 1) * n][:, fine], e[:, fine])


@pytest.mark.parametrize("source", ["logical", "tiles"])
def test_bf16_large_scales_in_a_layer(oracle, hm, device, source):
    # Up weights of about 2^120 and down weights of about 2^-100 (one matrix with large scales makes the layer take their
    # dequantization), a K range that splits, group 128, through both halves of the layer.
    rng = np.random.default_rng(325)
    hidden, inter, g, m = 2048, 256, 128, 40
    mats = [list(oracle.random_weights(rng, *s, g, "bf16")) for s in ((hidden, inter), (hidden, inter), (inter, hidden))]
    for i, e in ((1, 119), (2, -100)):
        mats[i][1] = _any_scales(rng, oracle, mats[i][1].shape, e, e + 1)[0]
    x64, x = make_x(oracle, rng, m, hidden, "bf16", device, scale=2.0 ** -4)
    if source == "logical":
        layer = hm.FfnLayer.from_logical(*(logical_to_device(t, "bf16", device) for t in mats), g, dtype=torch.bfloat16)
    else:
        packed = [torch.from_numpy(hm.pack_w4a16(q, s, z.astype(np.int8))).to(device) for q, s, z in mats]
        layer = hm.FfnLayer.from_tiles(*packed, hidden, inter, dtype=torch.bfloat16)
    act = layer.gate_up(x)
    y = layer.down(act)
    torch.cuda.synchronize()
    wg, wu, wd = (oracle.weights_f64(*t, g, "bf16") for t in mats)
    gate = x64 @ wg
    ref = gate / (1 + np.exp(-gate)) * (x64 @ wu)
    assert np.abs(ref).max() > 2.0 ** 115
    assert_close(oracle, host_f64(act) * 2.0 ** -118, ref * 2.0 ** -118, "bf16", "gate_up with large scales")
    assert_close(oracle, host_f64(y), host_f64(act) @ wd, "bf16", "down of the same layer")


@pytest.mark.parametrize("group", [32, 128])
@pytest.mark.parametrize("m,k,col,n", [(17, 4096, 0, 640), (40, 1280, 128, 256), (130, 4096, 256, 384), (300, 2176, 0, 640)])
def test_bf16_large_scales_forms(hm, device, m, k, col, n, group):
    # The large scales' kernel on blocks of a matrix, column ranges, strided rows, K splits and as either share of a K-split pair.
    # Integer activations times 2^-40 and scales of 2^115 .. 2^120: every sum is exact in fp32, so the output is the exact
    # result's rounding.
    gen = torch.Generator(device="cuda")
    gen.manual_seed(328 + m)
    rows, cols = 4096, 640
    mats, dense = [], []
    for lo, hi in ((115, 121), (-8, -4)):
        q = torch.randint(0, 16, (rows, cols), dtype=torch.uint8, device=device, generator=gen)
        z = torch.randint(0, 17, (rows // group, cols), dtype=torch.uint8, device=device, generator=gen)
        s = torch.exp2(torch.randint(lo, hi, (rows // group, cols), device=device, generator=gen).double()).to(torch.bfloat16)
        mats.append(hm.RepackedMatrix.from_logical(q, s, z, group, dtype=torch.bfloat16))
        dense.append(((q.view(-1, group, cols).double() - z.view(-1, 1, cols).double()) * s.view(-1, 1, cols).double()).view(rows, cols))
    wide = torch.randint(-2, 3, (m, k + 64), device=device, generator=gen).to(torch.bfloat16) * 2.0 ** -40
    x = wide[:, :k]
    ref = (x.double() @ dense[0][:k, col:col + n]).to(torch.bfloat16)
    frame = torch.full((m + 1, n + 16), 7.0, dtype=torch.bfloat16, device=device)
    y = frame[:m, :n]
    hm.packed_linear(y, x, mats[0], k=k, n=n, col_begin=col)
    torch.cuda.synchronize()
    assert torch.equal(y, ref)
    y.fill_(7.0)
    assert bool((frame == 7.0).all())
    both = torch.cat([x, x], dim=1)
    small = (x.double() @ dense[1][:k, :n]).to(torch.bfloat16)
    large = (x.double() @ dense[0][:k, :n]).to(torch.bfloat16)
    for pair in (mats, mats[::-1]):
        out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=device)
        hm.packed_linear_k_split(out, both, *pair, k0=k, k1=k, n=n)
        torch.cuda.synchronize()
        assert torch.equal(out, large + small)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("k,n,group", [(1152, 384, 32), (1408, 128, 64), (2688, 1024, 128), (1024, 6144, 64)])
def test_tile_edges(oracle, hm, device, k, n, group, dtype):
    # Rows on both sides of 32 to 128 in steps of 16 and beyond, in a frame that has to stay untouched; 9, 11 and 21 K tiles do
    # not divide into the K groups. These matrices mostly take the 32- and 48-row tiles (the others: test_gpu_gemm_plans.py).
    # The second share of a K-split pair adds into its output through the same tiles.
    rng = np.random.default_rng(330 + k + n)
    w_np = oracle.random_weights(rng, k, n, group, dtype)
    w = hm.RepackedMatrix.from_logical(*logical_to_device(w_np, dtype, device), group, dtype=TORCH[dtype])
    wf = oracle.weights_f64(*w_np, group, dtype)
    for m in (17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129, 177, 225, 257, 385):
        x64, x = make_x(oracle, rng, m, k, dtype, device)
        frame = torch.full((m + 2, n + 32), 7.0, dtype=TORCH[dtype], device=device)
        y = frame[1:m + 1, 16:n + 16]
        hm.packed_linear(y, x, w)
        torch.cuda.synchronize()
        assert_close(oracle, host_f64(y), x64 @ wf, dtype, f"linear {k}x{n} g={group} M={m}")
        y2 = torch.empty((m, n), dtype=TORCH[dtype], device=device)
        hm.packed_linear_k_split(y2, torch.cat([x, x], dim=1), w, w)
        torch.cuda.synchronize()
        assert torch.equal(y2, y + y), (k, n, m)
        frame[1:m + 1, 16:n + 16] = 7.0
        assert bool((frame == 7.0).all()), (k, n, m)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("hidden,inter,group", [(1152, 1408, 128), (2048, 8192, 64)])
def test_tile_edges_fused(oracle, hm, device, hidden, inter, group, dtype):
    # The fused gate_up, SwiGLU after the K groups' exchange.
    rng = np.random.default_rng(350 + hidden)
    ws = [oracle.random_weights(rng, hidden, inter, group, dtype), oracle.random_weights(rng, hidden, inter, group, dtype),
          oracle.random_weights(rng, inter, hidden, group, dtype)]
    layer = hm.FfnLayer.from_logical(*(logical_to_device(t, dtype, device) for t in ws), group, dtype=TORCH[dtype])
    wg, wu = (oracle.weights_f64(*t, group, dtype) for t in ws[:2])
    for m in (17, 33, 64, 80, 97, 128, 160, 200, 320):
        x64, x = make_x(oracle, rng, m, hidden, dtype, device)
        act = layer.gate_up(x)
        torch.cuda.synchronize()
        g = x64 @ wg
        assert_close(oracle, host_f64(act), g / (1 + np.exp(-g)) * (x64 @ wu), dtype, f"gate_up {hidden}x{inter} M={m}")
