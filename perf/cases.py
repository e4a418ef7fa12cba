"""The calls a user of this package makes, over the sizes they make them at: whole MoE layers from one decode token to a
long prefill, the drop-in expert op in the reference's argument form, the dense layers, and the two 16-bit arithmetics.

A case is a dict of plain values.  "kind" says which entry point is called:

  layer   `FusedMoE(x)`: router, routing, permutation, both grouped products, weighted sum (+ shared expert)
  op      `torch.ops.my_ops.fused_moe_fused_experts`: the reference's op on given routing, [T, K, H] or [T, H] output
  mm/mlp  `torch.ops.my_ops.mm_w8a16_dq_forward` / `mlp_w8a16_dq_forward`: block-scaled dense layers
  w8a16   `fused_experts_w8a16`: FP8 weights against bf16 activations
  bf16    `fused_experts_bf16`: un-quantised experts
"""
import importlib.util
import math
import os
import sys

import torch


def _package():
    """The package directory `torch-tpu_amd/` of the working folder, under its importable name."""
    name = "torch_tpu_amd"
    if name not in sys.modules:
        folder = os.path.join(os.getcwd(), "torch-tpu_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
    return sys.modules[name]


# Layer shapes: the four workloads of bench.py.  zipf: expert popularity ~ rank^-zipf, `empty` experts never chosen.
LAYERS = {
    "deepseek_v3": dict(H=7168, I=2048, E=256, K=8, shared=True, route="sigmoid", n_groups=8, topk_groups=4, scale=2.5),
    "mixtral": dict(H=4096, I=14336, E=8, K=2, shared=False, route="softmax", n_groups=1, topk_groups=1, scale=1.0),
    "qwen3": dict(H=2048, I=768, E=128, K=8, shared=False, route="softmax", n_groups=1, topk_groups=1, scale=1.0),
    "toy": dict(H=256, I=512, E=8, K=2, shared=False, route="softmax", n_groups=1, topk_groups=1, scale=1.0),
}
DENSE_MM = [(7168, 1536), (2048, 7168), (16384, 1024), (4096, 4096), (4096, 28672), (7168, 7168), (7168, 36864)]   # K, N
DENSE_MLP = [(7168, 18432), (4096, 14336), (7168, 2048)]                                                          # H, I


def _layer(shape, T, skew=False):
    return dict(kind="layer", T=T, skew=skew, **LAYERS[shape])


def _experts(kind, shape, T, **more):
    return dict(kind=kind, T=T, **{k: LAYERS[shape][k] for k in ("H", "I", "E", "K")}, **more)


def listed():
    return [
        # one user's next token: a chain of small launches around 0.4 GB of weights
        dict(name="layer_deepseek_t1", **_layer("deepseek_v3", 1)),
        # a decode batch: most experts touched by a row or two, the weight stream counts
        dict(name="layer_deepseek_t32", **_layer("deepseek_v3", 32)),
        # a short prompt or a chunk of one, ragged: every expert holds about nineteen rows
        dict(name="layer_deepseek_t613", **_layer("deepseek_v3", 613)),
        # the headline prefill: 128 rows per expert on average
        dict(name="layer_deepseek_t4096", **_layer("deepseek_v3", 4096)),
        # few wide experts, a thousand rows each: the matrix cores count
        dict(name="layer_mixtral_t4096", **_layer("mixtral", 4096)),
        # many narrow experts, a long prompt under a skewed load with empty experts
        dict(name="layer_qwen3_t16384_skewed", **_layer("qwen3", 16384, True)),
        # the drop-in op as the reference's callers use it at decode: per-slot output, routing given
        dict(name="op_qwen3_t20_per_slot", **_experts("op", "qwen3", 20, weighted=False)),
        # an attention projection at decode, the smallest call there is
        dict(name="mm_7168_1536_m32", kind="mm", M=32, K=7168, N=1536),
        # the same projection over a prefill, a ragged batch
        dict(name="mm_7168_1536_m4001", kind="mm", M=4001, K=7168, N=1536),
        # the dense MLP of the first layers on a chunk of prompt, ragged
        dict(name="mlp_7168_18432_m300", kind="mlp", M=300, H=7168, I=18432),
        # the reference's own arithmetic on FP8 weights, a mixed batch of decode and chunks
        dict(name="w8a16_mixtral_t333", **_experts("w8a16", "mixtral", 333, weighted=True)),
        # un-quantised experts over a prompt
        dict(name="bf16_qwen3_t2048", **_experts("bf16", "qwen3", 2048, weighted=True)),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "op", "mm", "mm", "mlp", "w8a16", "bf16"])
    if kind == "layer":
        shape = rng.choice(["deepseek_v3", "mixtral", "qwen3", "toy", "any"])
        if shape != "any":
            most = {"deepseek_v3": 4096, "mixtral": 4096, "qwen3": 16384, "toy": 16384}[shape]
            return _layer(shape, _log_int(rng, 1, most), shape == "qwen3" and rng.random() < 0.5)
        # a layer of no particular model: any whole number of 128-blocks
        E = rng.randint(8, 160)
        c = dict(H=128 * rng.randint(8, 40), I=128 * rng.randint(2, 16), E=E, K=rng.randint(1, 8),
                 shared=rng.random() < 0.3, route="softmax", n_groups=1, topk_groups=1, scale=1.0)
        return dict(kind="layer", T=_log_int(rng, 1, 4096), skew=rng.random() < 0.3, **c)
    if kind == "op":
        c = _experts("op", rng.choice(["qwen3", "qwen3", "toy"]), _log_int(rng, 1, 4096), weighted=rng.random() < 0.5)
        if rng.random() < 0.3:
            c["I"] = 8 * rng.randint(40, 190)          # a ragged last block
        return c
    if kind == "mm":
        K, N = rng.choice(DENSE_MM)
        if rng.random() < 0.3:
            N += rng.choice([-48, -16, 16, 64])
        return dict(kind="mm", M=_log_int(rng, 1, 4096), K=K, N=N)
    if kind == "mlp":
        H, I = rng.choice(DENSE_MLP)
        return dict(kind="mlp", M=_log_int(rng, 1, 4000), H=H, I=I)
    shape = rng.choice(["mixtral", "qwen3", "toy"]) if kind == "w8a16" else rng.choice(["qwen3", "toy"])
    return _experts(kind, shape, _log_int(rng, 1, 2048), weighted=rng.random() < 0.5)


# ---------------------------------------------------------------------------------------------- inputs
DEV = "cuda"


def _gen(seed, part):
    return torch.Generator(device=DEV).manual_seed(1000003 * (seed % (1 << 40)) + part)


def _bf16(seed, part, *shape, std=1.0):
    return (torch.randn(*shape, generator=_gen(seed, part), device=DEV) * std).to(torch.bfloat16)


def _quantised(seed, part, *shape):
    """Row-major weights ~ N(0, 0.02) as a checkpoint holds them: e4m3fn codes and bf16 scales per 128 x 128 block, the
    last block of a side that 128 does not divide partial."""
    n, k = shape[-2:]
    codes = (torch.randn(*shape, generator=_gen(seed, part), device=DEV) * 105.0).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
    lead = shape[:-2]
    scale = 0.02 / 105.0 * (0.9 + 0.2 * torch.rand(*lead, -(-n // 128), -(-k // 128), generator=_gen(seed, part + 1), device=DEV))
    return codes, scale.to(torch.bfloat16)


def _routing(seed, T, E, K):
    """Distinct experts per token, some more popular than others, and weights that add up to one, bf16 as callers hold them."""
    popular = 0.5 * torch.randn(E, generator=_gen(seed, 31), device=DEV)
    w, ids = (popular + torch.randn(T, E, generator=_gen(seed, 32), device=DEV)).topk(K, dim=1)
    return ids.to(torch.int32), torch.softmax(w, dim=1).to(torch.bfloat16)


def prepare(case, seed):
    pkg = _package()
    c = dict(case)
    seed = int(seed)
    if c["kind"] in ("layer", "w8a16", "bf16", "op"):
        T, H, I, E, K = c["T"], c["H"], c["I"], c["E"], c["K"]
    if c["kind"] == "layer":
        w13 = pkg.synthetic_weights(E, 2 * I, H, DEV, 8 * seed + 1)
        w2 = pkg.synthetic_weights(E, H, I, DEV, 8 * seed + 2)
        shared = None
        if c["shared"]:
            shared = (*pkg.synthetic_weights(1, 2 * I, H, DEV, 8 * seed + 3), *pkg.synthetic_weights(1, H, I, DEV, 8 * seed + 4))
        bias = None
        if c["skew"]:
            rank = torch.randperm(E, generator=_gen(seed, 5), device=DEV)
            bias = -1.2 * torch.log(rank.float() + 1)
            bias[rank >= max(K, E - E // 10)] = -1e9             # a tenth of the experts is never chosen
        elif c["route"] == "sigmoid":
            bias = 0.01 * torch.randn(E, generator=_gen(seed, 5), device=DEV)      # the correction bias of the selection
        moe = pkg.FusedMoE(_bf16(seed, 6, E, H, std=0.02), *w13, *w2, top_k=K, mode=c["route"], bias=bias,
                           n_groups=c["n_groups"], topk_groups=c["topk_groups"], renorm=True, scale=c["scale"], shared=shared)
        return dict(kind="layer", moe=moe, x=_bf16(seed, 7, T, H))
    if c["kind"] == "op":
        (gate, gs), (up, us), (down, ds) = (_quantised(seed, 10 + 2 * i, E, I, H) for i in range(3))
        ids, rw = _routing(seed, T, E, K)
        out = torch.empty((T, H) if c["weighted"] else (T, K, H), dtype=torch.bfloat16, device=DEV)
        s = dict(kind="op", out=out, x=_bf16(seed, 7, T, H), w=(gate, up, down, gs, us, ds), ids=ids, rw=rw, E=E, K=K)
        # the op lays the weights out at its first call; a serving program makes that one when it loads
        run(dict(s, out=torch.empty((1, *out.shape[1:]), dtype=torch.bfloat16, device=DEV), x=s["x"][:1], ids=ids[:1], rw=rw[:1]))
        return s
    if c["kind"] == "mm":
        w, scale = _quantised(seed, 10, c["N"], c["K"])
        s = dict(kind="mm", x=_bf16(seed, 7, c["M"], c["K"]), w=(w, scale),
                 out=torch.empty(c["M"], c["N"], dtype=torch.bfloat16, device=DEV))
        run(dict(s, x=s["x"][:1], out=torch.empty(1, c["N"], dtype=torch.bfloat16, device=DEV)))
        return s
    if c["kind"] == "mlp":
        H, I = c["H"], c["I"]
        (gate, gs), (up, us), (down_t, ds) = (_quantised(seed, 10 + 2 * i, I, H) for i in range(3))
        s = dict(kind="mlp", x=_bf16(seed, 7, c["M"], H), w=(gate, up, down_t, gs, us, ds),
                 out=torch.empty(c["M"], H, dtype=torch.bfloat16, device=DEV))
        run(dict(s, x=s["x"][:1], out=torch.empty(1, H, dtype=torch.bfloat16, device=DEV)))
        return s
    ids, rw = _routing(seed, T, E, K)
    ws = torch.empty(pkg.ops.fused_experts_bf16_workspace_bytes(T, H, I, E, K), dtype=torch.uint8, device=DEV)
    s = dict(kind=c["kind"], x=_bf16(seed, 7, T, H), ids=ids, rw=rw.float() if c["weighted"] else None, ws=ws)
    if c["kind"] == "w8a16":
        s["w"] = (*pkg.synthetic_weights(E, 2 * I, H, DEV, 8 * seed + 1), *pkg.synthetic_weights(E, H, I, DEV, 8 * seed + 2))
    else:
        s["w"] = (pkg.pack_weights(_bf16(seed, 8, E, 2 * I, H, std=0.02)), pkg.pack_weights(_bf16(seed, 9, E, H, I, std=0.02)))
    return s


def run(state):
    s = state
    if s["kind"] == "layer":
        return s["moe"](s["x"])
    my_ops = torch.ops.my_ops
    if s["kind"] == "op":
        gate, up, down, gs, us, ds = s["w"]
        return my_ops.fused_moe_fused_experts(s["out"], s["x"], None, None, gate, up, down, gs, us, ds, s["ids"], s["rw"],
                                              None, None, None, 128, s["E"], s["K"], False, 0, 0, None, None, None, False)
    if s["kind"] == "mm":
        return my_ops.mm_w8a16_dq_forward(s["x"], *s["w"], s["out"], 128)
    if s["kind"] == "mlp":
        return my_ops.mlp_w8a16_dq_forward(s["x"], *s["w"], s["out"], 128)
    pkg = _package()
    if s["kind"] == "w8a16":
        return pkg.fused_experts_w8a16(s["x"], *s["w"], s["ids"], s["rw"], workspace=s["ws"])
    return pkg.fused_experts_bf16(s["x"], *s["w"], s["ids"], s["rw"], workspace=s["ws"])


def work(case):
    """Every touched expert's weights and scales read once, the activations read and the output written once."""
    c = dict(case)
    if c["kind"] == "mm":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": N * K + 2.0 * M * (K + N), "flops": 2.0 * M * K * N}
    if c["kind"] == "mlp":
        M, H, I = c["M"], c["H"], c["I"]
        return {"bytes": 3.0 * H * I + 4.0 * M * H, "flops": 6.0 * M * H * I}
    T, H, I, E, K = c["T"], c["H"], c["I"], c["E"], c["K"]
    usable = E - E // 10 if c.get("skew") else E
    touched = usable * (1.0 - (1.0 - min(K, usable) / usable) ** T)      # expected, under even routing
    shared = 1 if c.get("shared") else 0
    per_weight = 2 if c["kind"] == "bf16" else 1
    per_slot = c["kind"] != "layer" and not c["weighted"]
    io = 2.0 * T * H * (1 + (K if per_slot else 1))
    router = 2.0 * E * H if c["kind"] == "layer" else 0.0
    return {"bytes": (touched + shared) * 3.0 * H * I * per_weight + io + router,
            "flops": 6.0 * H * I * T * (K + shared) + (2.0 * T * E * H if c["kind"] == "layer" else 0.0)}


def tolerance(case):
    """About four times what the path shows against itself with every sum in 64 bits.  Quantised intermediates: rel 0.0095 to
    0.016, max 0.10 to 0.15 (an element of the intermediate on a rounding boundary lands on the neighbouring e4m3 code).
    A single quantised product: rel 0.0036, max 0.026.  16-bit arithmetic: rel 0.0017, max 0.010 (the bf16 result)."""
    kind = case["kind"]
    if kind == "mm":
        return {"rel": 0.012, "max": 0.1}
    if kind in ("w8a16", "bf16"):
        return {"rel": 0.006, "max": 0.04}
    return {"rel": 0.03, "max": 0.5}
