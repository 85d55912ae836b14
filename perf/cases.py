"""Performance cases of the W4A16 SwiGLU FFN engine.

A pass is the weight-bound part of one model step: every layer of a model (or a run of layers long enough that the
weights do not sit in the 256 MB Infinity Cache, as those of a whole model never do) called once through the public
operators, each layer on the input the rest of the model hands it. The kinds:

  ffn      GpuFfnModel.forward of each layer: y = (SiLU(x Wg) * (x Wu)) Wd
  stack    FfnLayer.block_forward of each layer in turn on one residual stream: x += FFN(RMSNorm(x) * w)
  linear   packed_linear of each layer's attention projection (Q, K and V side by side)
  k_split  packed_linear_k_split of each layer's down projection, kept as a pair of matrices over K

Rows run from one (decode of one sequence) over a few to some tens (batched decode, verification of drafted tokens,
short prompts) to 2048 (a prompt chunk); layer shapes are those of Llama-3.2-1B, Llama-3-8B and Qwen2.5-14B and others
between them; groups of 128, 64 and 32; fp16 and bf16. Weights are uniform int4 with scales U(0.001, 0.02) and int4
zero points, activations N(0, 1).
"""

import math

import torch

import heteromega_amd as hm

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
_CACHE_BYTES = 300e6  # weights of a pass at up to 512 rows: more than the Infinity Cache holds
_LARGEST_FLOPS = 1.45e12


def _ffn(name, kind, rows, hidden, inter, group, dtype, layers):
    return {"name": name, "kind": kind, "rows": rows, "hidden": hidden, "inter": inter, "group": group, "dtype": dtype, "layers": layers}


def _linear(name, rows, k, n, group, dtype, layers):
    return {"name": name, "kind": "linear", "rows": rows, "k": k, "n": n, "group": group, "dtype": dtype, "layers": layers}


def _k_split(name, rows, k0, k1, n, group, dtype, layers):
    return {"name": name, "kind": "k_split", "rows": rows, "k0": k0, "k1": k1, "n": n, "group": group, "dtype": dtype, "layers": layers}


def listed():
    return [
        # One decoded token's attention projections, Llama-3-8B: the smallest calls, one short launch each.
        _linear("qkv_8b_m1_fp16", 1, 4096, 6144, 128, "fp16", 24),
        # One decoded token through the FFNs of Llama-3.2-1B: small layers, launches count.
        _ffn("ffn_1b_m1_fp16", "ffn", 1, 2048, 8192, 128, "fp16", 16),
        # One decoded token through all 32 FFN blocks of Llama-3-8B, norm and residual included: a whole call.
        _ffn("stack_8b_m1_fp16", "stack", 1, 4096, 14336, 128, "fp16", 32),
        # One decoded token, Qwen2.5-14B shape (odd multiples of the tiles), groups of 64, bf16.
        _ffn("ffn_14b_g64_m1_bf16", "ffn", 1, 5120, 13824, 64, "bf16", 4),
        # Decode of a batch of four.
        _ffn("ffn_8b_m4_bf16", "ffn", 4, 4096, 14336, 128, "bf16", 4),
        # Decode of a batch of sixteen.
        _ffn("ffn_8b_m16_fp16", "ffn", 16, 4096, 14336, 128, "fp16", 4),
        # A larger decode batch or a short question: an odd row count past the decode kernels.
        _ffn("ffn_8b_m37_fp16", "ffn", 37, 4096, 14336, 128, "fp16", 4),
        # A short prompt, Qwen2.5-14B shape, groups of 64, bf16.
        _ffn("ffn_14b_g64_m100_bf16", "ffn", 100, 5120, 13824, 64, "bf16", 4),
        # The down projection of a pre-saved K-split pair with unequal shares, a prompt of 200 tokens.
        _k_split("k_split_8b_m200_bf16", 200, 4096, 10240, 4096, 128, "bf16", 10),
        # A prompt of 300 tokens through all 16 FFN blocks of Llama-3.2-1B: a whole call.
        _ffn("stack_1b_m300_bf16", "stack", 300, 2048, 8192, 128, "bf16", 16),
        # A prompt of 512 tokens, bf16.
        _ffn("ffn_8b_m512_bf16", "ffn", 512, 4096, 14336, 128, "bf16", 4),
        # A prompt chunk of 2048 tokens: the largest call.
        _ffn("ffn_8b_m2048_fp16", "ffn", 2048, 4096, 14336, 128, "fp16", 2),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choice(("ffn", "ffn", "ffn", "stack", "linear", "linear", "k_split"))
    rows = _log_int(rng, 1, 2048)
    group = rng.choice((128, 128, 128, 64, 32))
    dtype = rng.choice(("fp16", "bf16"))
    hidden = 128 * rng.randint(16, 40)
    if kind in ("ffn", "stack"):
        case = _ffn("", kind, rows, hidden, 128 * _log_int(rng, 48, 112), group, dtype, 1)
    elif kind == "linear":
        # past 16 rows the operator takes columns in multiples of 128, up to it of 16
        n = 128 * _log_int(rng, 8, 56) if rows > 16 else 16 * _log_int(rng, 64, 448)
        case = _linear("", rows, hidden, n, group, dtype, 1)
    else:
        tiles = _log_int(rng, 48, 112)
        k0 = rng.randint(8, tiles - 8)
        case = _k_split("", rows, 128 * k0, 128 * (tiles - k0), hidden, group, dtype, 1)
    one = work(case)
    layers = min(32, max(2, math.ceil(_CACHE_BYTES / _weight_bytes(case)))) if rows <= 512 else 2
    case["layers"] = max(1, min(layers, int(_LARGEST_FLOPS // one["flops"])))
    del case["name"]
    return case


def _shapes(case):
    """[(K, N)] of the matrices of one layer, in the order they are made."""
    if case["kind"] in ("ffn", "stack"):
        h, i = case["hidden"], case["inter"]
        return [(h, i), (h, i), (i, h)]
    if case["kind"] == "linear":
        return [(case["k"], case["n"])]
    return [(case["k0"], case["n"]), (case["k1"], case["n"])]


def _in_out(case):
    """Columns of one layer's input and output."""
    if case["kind"] in ("ffn", "stack"):
        return case["hidden"], case["hidden"]
    if case["kind"] == "linear":
        return case["k"], case["n"]
    return case["k0"] + case["k1"], case["n"]


def _weight_bytes(case):
    """int4 weights, a 2-byte scale and a 1-byte zero point per column and group."""
    return sum(k * n // 2 + k // case["group"] * n * 3 for k, n in _shapes(case))


def _layer_gen(seed, layer):
    gen = torch.Generator(device="cuda")
    gen.manual_seed((seed * 1009 + layer) % (1 << 62))
    return gen


def _logical(case, gen):
    """One layer's matrices as (q [K, N], scales [K / group, N], zeros [K / group, N])."""
    g, dtype = case["group"], _DTYPES[case["dtype"]]
    mats = []
    for k, n in _shapes(case):
        q = torch.randint(0, 16, (k, n), dtype=torch.uint8, device="cuda", generator=gen)
        s = (torch.rand((k // g, n), device="cuda", generator=gen) * 0.019 + 0.001).to(dtype)
        z = torch.randint(0, 16, (k // g, n), dtype=torch.uint8, device="cuda", generator=gen)
        mats.append((q, s, z))
    return mats


def _input(case, gen, cols):
    return torch.randn((case["rows"], cols), device="cuda", generator=gen).to(_DTYPES[case["dtype"]])


def _norm_weight(case, gen):
    return (1.0 + 0.1 * torch.randn((case["hidden"],), device="cuda", generator=gen)).to(_DTYPES[case["dtype"]])


def prepare(case, seed):
    dtype, g, rows = _DTYPES[case["dtype"]], case["group"], case["rows"]
    kin, kout = _in_out(case)
    state = {"kind": case["kind"], "layers": case["layers"], "x": [], "y": [], "w": []}
    if case["kind"] == "ffn":
        state["model"] = hm.GpuFfnModel(dtype)
    if case["kind"] == "stack":
        state["x0"] = _input(case, _layer_gen(seed, -1), kin)
        state["x"] = torch.empty_like(state["x0"])
        state["norm"] = []
    for layer in range(case["layers"]):
        gen = _layer_gen(seed, layer)
        mats = _logical(case, gen)
        if case["kind"] == "ffn":
            state["model"].add_layer_logical(*mats, g)
        elif case["kind"] == "stack":
            state["w"].append(hm.FfnLayer.from_logical(*mats, g, dtype=dtype))
            state["norm"].append(_norm_weight(case, gen))
            continue
        else:
            state["w"].append([hm.RepackedMatrix.from_logical(*m, g, dtype=dtype) for m in mats])
        state["x"].append(_input(case, gen, kin))
        state["y"].append(torch.empty((rows, kout), dtype=dtype, device="cuda"))
    # The scratch that a serving program keeps for its projections (the FFN layers keep their own).
    if case["kind"] == "linear":
        state["ws"] = torch.empty(state["w"][0][0].workspace_bytes(rows) + 256, dtype=torch.uint8, device="cuda")
    return state


def run(state):
    kind = state["kind"]
    if kind == "ffn":
        for layer in range(state["layers"]):
            state["model"].forward(layer, state["x"][layer], state["y"][layer])
        return state["y"]
    if kind == "stack":
        # the residual stream starts from the embeddings
        x = state["x"].copy_(state["x0"])
        for layer in range(state["layers"]):
            state["w"][layer].block_forward(x, state["norm"][layer])
        return x
    if kind == "linear":
        for layer in range(state["layers"]):
            hm.packed_linear(state["y"][layer], state["x"][layer], state["w"][layer][0], workspace=state["ws"])
        return state["y"]
    for layer in range(state["layers"]):
        hm.packed_linear_k_split(state["y"][layer], state["x"][layer], *state["w"][layer])
    return state["y"]


def work(case):
    kin, kout = _in_out(case)
    rows, layers = case["rows"], case["layers"]
    io = rows * (kin + kout) * 2
    flops = sum(2 * rows * k * n for k, n in _shapes(case))
    if case["kind"] == "stack":  # the residual stream enters and leaves once
        return {"bytes": layers * (_weight_bytes(case) + 2 * case["hidden"]) + io, "flops": layers * flops}
    return {"bytes": layers * (_weight_bytes(case) + io), "flops": layers * flops}


def tolerance(case):
    # One layer against 64 bits: the output's rounding, the SwiGLU activation's and (past the decode kernels) the
    # weights' once each. A stack carries each layer's roundings through all that follow.
    if case["kind"] == "stack":
        return {"rel": 1.2e-2} if case["dtype"] == "fp16" else {"rel": 8e-2}
    return {"rel": 1.5e-3, "max": 1e-2} if case["dtype"] == "fp16" else {"rel": 1.2e-2, "max": 8e-2}


def exact(case, seed):
    g = case["group"]

    def dense(mat):
        q, s, z = mat
        k, n = q.shape
        w = (q.view(k // g, g, n).double() - z.view(k // g, 1, n).double()) * s.view(k // g, 1, n).double()
        return w.view(k, n)

    def ffn(x, mats):
        gate = x @ dense(mats[0])
        up = x @ dense(mats[1])
        return (gate / (1.0 + torch.exp(-gate)) * up) @ dense(mats[2])

    kin, _ = _in_out(case)
    if case["kind"] == "stack":
        x = _input(case, _layer_gen(seed, -1), kin).double()
        for layer in range(case["layers"]):
            gen = _layer_gen(seed, layer)
            mats = _logical(case, gen)
            normed = x * torch.rsqrt((x * x).mean(dim=1, keepdim=True) + 1e-5) * _norm_weight(case, gen).double()
            x = x + ffn(normed, mats)
        return x
    out = []
    for layer in range(case["layers"]):
        gen = _layer_gen(seed, layer)
        mats = _logical(case, gen)
        x = _input(case, gen, kin).double()
        if case["kind"] == "ffn":
            out.append(ffn(x, mats))
        elif case["kind"] == "linear":
            out.append(x @ dense(mats[0]))
        else:
            k0 = case["k0"]
            out.append(x[:, :k0] @ dense(mats[0]) + x[:, k0:] @ dense(mats[1]))
    return out
