"""The workloads this package's speed is judged by: W4A16 linears as a model runs them.

Layer shapes are those of the benchmark and the tests (the Llama-3-8B and -70B shaped linears)
and generic odd sizes; activations are N(0, 1), int4 codes uniform, scales |N(0, 0.02)| + 1e-3,
as in the benchmark.  Every case goes through a public entry point: the operators of
`pulsar_amd.ops`, the modules of `pulsar_amd.linear` and the graph runner of `pulsar_amd.stack`.
"""

from __future__ import annotations

import math

import torch

from pulsar_amd import ops
from pulsar_amd.linear import W4A16Linear, W4A16SiluGate
from pulsar_amd.stack import LLAMA3_8B_LINEARS, W4A16LinearStack, fuse_layers

DEVICE = "cuda:0"

# (K, N) of the layers the benchmark and the tests run
LAYERS_8B = ((4096, 4096), (4096, 6144), (4096, 28672), (14336, 4096))
LAYERS_70B = ((8192, 8192), (8192, 10240), (28672, 8192))


def _case(kind: str, m: int, k: int, n: int, group: int = 128, dtype: str = "f16", zp: bool = False,
          act: bool = False, layers: int = 1) -> dict:
    return {"kind": kind, "m": m, "k": k, "n": n, "group": group, "dtype": dtype, "zp": zp, "act": act,
            "layers": layers}


def listed() -> list[dict]:
    named = {
        # one eager operator call of the smallest layer for one token: launch and host latency
        "call_o_m1": _case("marlin", 1, 4096, 4096, dtype="bf16"),
        # the linears of four decoder layers as one graph, the way a decode step replays them:
        # one sequence, a small batch, and the batch of 32 the stack is benchmarked at.  Four
        # layers hold 450 MB, so the weights stream from HBM as in a whole model.
        "stack_m1": _case("stack", 1, 4096, 14336, layers=4),
        "stack_m16": _case("stack", 16, 4096, 14336, layers=4),
        "stack_m32": _case("stack", 32, 4096, 14336, layers=4),
        # a checkpoint's packed weight used as it is, without the one-time repack
        "packed_qkv_m4": _case("packed", 4, 4096, 6144),
        # a 70B layer of a GPTQ checkpoint with zero points and act-order, a few sequences
        "act_order_qkv_m8": _case("linear", 8, 8192, 10240, zp=True, act=True),
        # the gated MLP of a serving batch of 64 sequences, in the engine's bf16
        "silu_gate_m64": _case("silu", 64, 4096, 14336, dtype="bf16"),
        # a prompt chunk whose sizes divide nothing: ragged rows, columns and K, groups of 64
        "ragged_m197": _case("linear", 197, 4160, 5000, group=64, zp=True),
        # a short prompt through down_proj in bf16, on the reference's operator
        "prefill_down_m1024": _case("marlin", 1024, 14336, 4096, dtype="bf16"),
        # a long prompt through gate|up, the largest GEMM of the layer
        "prefill_gate_up_m4096": _case("linear", 4096, 4096, 28672),
        # a prompt chunk on a packed weight used as it is
        "packed_o_m512": _case("packed", 512, 4096, 4096, dtype="bf16"),
        # loading: down_proj of an act-order checkpoint into the kernels' layout
        "load_act_order_down": _case("repack_gptq", 0, 14336, 4096, act=True),
    }
    return [dict(c, name=name) for name, c in named.items()]


# 2 M N K of a drawn case: below a third of the largest listed one, since small quant groups
# run on a kernel of about half the speed
MAX_DRAWN_FLOPS = 0.3e12


def draw(rng) -> dict:
    kind = rng.choices(("linear", "marlin", "silu", "stack", "packed", "repack_gptq", "repack_packed"),
                       (8, 4, 3, 3, 3, 1, 1))[0]
    if kind == "stack":
        return _case("stack", min(64, max(1, round(2 ** rng.uniform(-0.5, 6)))), 4096, 14336,
                     layers=rng.randint(2, 4))
    group = rng.choices((128, 64, 32), (6, 2, 1))[0]
    dtype = rng.choice(("f16", "bf16"))
    if rng.random() < 0.5:
        k, n = rng.choice(LAYERS_8B + LAYERS_70B)
    else:  # any K of whole groups, any N of whole zero-point words
        k = group * max(1, round(2 ** rng.uniform(math.log2(512), math.log2(14336)) / group))
        n = 8 * round(2 ** rng.uniform(math.log2(512), math.log2(28672)) / 8)
    if kind == "silu":
        n = max(64, n // 2 // 64 * 64)  # columns of gate and of up
    m = max(1, round(2 ** rng.uniform(-0.5, 12)))
    flops = 2 * m * k * n * (2 if kind == "silu" else 1)
    if flops > MAX_DRAWN_FLOPS:
        m = max(1, int(m * MAX_DRAWN_FLOPS / flops))
    if kind.startswith("repack"):
        m = 0
    gptq = kind in ("linear", "silu", "repack_gptq")
    return _case(kind, m, k, n, group, dtype, zp=gptq and kind != "repack_gptq" and rng.random() < 0.5,
                 act=gptq and rng.random() < (0.5 if kind == "repack_gptq" else 0.3))


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _words(rows: int, cols: int, gen) -> torch.Tensor:
    return torch.randint(-(2 ** 31), 2 ** 31, (rows, cols), dtype=torch.int32, device=DEVICE, generator=gen)


def _scales(rows: int, cols: int, gen) -> torch.Tensor:
    return (torch.randn(rows, cols, device=DEVICE, generator=gen) * 0.02).abs_().add_(1e-3).half()


def _x(case: dict, k: int, gen) -> torch.Tensor:
    dt = torch.float16 if case["dtype"] == "f16" else torch.bfloat16
    return torch.randn(case["m"], k, device=DEVICE, generator=gen).to(dt)


def _gptq(k: int, n: int, case: dict, gen) -> dict:
    """A GPTQ checkpoint's tensors of one [n, k] linear."""
    g = case["group"]
    t = {"qweight": _words(k // 8, n, gen), "scales": _scales(k // g, n, gen), "qzeros": None, "g_idx": None}
    if case["zp"]:
        t["qzeros"] = _words(k // g, n // 8, gen)
    if case["act"]:
        groups = torch.arange(k, device=DEVICE, dtype=torch.int32) // g
        t["g_idx"] = groups[torch.randperm(k, device=DEVICE, generator=gen)].contiguous()
    return t


def _packed(case: dict, gen) -> dict:
    """A compressed-tensors weight: int32 [N, K/8] and scales [N, K/G]."""
    k, n = case["k"], case["n"]
    return {"packed": _words(n, k // 8, gen), "scales": _scales(n, k // case["group"], gen)}


def _raw(case: dict, seed: int) -> dict:
    gen = _gen(seed)
    kind, k, n = case["kind"], case["k"], case["n"]
    if kind == "stack":
        layers = [{name: _gptq(lk, ln, case, gen) for name, lk, ln in LLAMA3_8B_LINEARS}
                  for _ in range(case["layers"])]
        return {"layers": layers, "x": _x(case, k, gen)}
    if kind == "silu":
        gate, up = _gptq(k, n, case, gen), _gptq(k, n, case, gen)
        up["g_idx"] = gate["g_idx"]  # gate and up read one input in one order
        return {"gate": gate, "up": up, "x": _x(case, k, gen)}
    t = _packed(case, gen) if kind in ("packed", "marlin", "repack_packed") else _gptq(k, n, case, gen)
    return {"w": t, "x": _x(case, k, gen)}


def _linear(t: dict, group: int) -> W4A16Linear:
    return W4A16Linear.from_gptq(t["qweight"], t["scales"], group, qzeros=t["qzeros"], g_idx=t["g_idx"])


def prepare(case: dict, seed: int) -> dict:
    raw, kind, g = _raw(case, seed), case["kind"], case["group"]
    if kind == "stack":
        layers = []
        for tensors in raw["layers"]:
            layer = []
            for name, _, _ in LLAMA3_8B_LINEARS:
                lin = _linear(tensors[name], g)
                lin.name = name
                layer.append(lin)
            layers.append(layer)
        stack = W4A16LinearStack(fuse_layers(layers, silu_gate=True), case["m"], g, DEVICE)
        stack.inputs[case["k"]].copy_(raw["x"])
        stack.capture()
        return {"kind": kind, "stack": stack}
    if kind == "linear":
        return {"kind": kind, "layer": _linear(raw["w"], g), "x": raw["x"]}
    if kind == "silu":
        layer = W4A16SiluGate.from_members(_linear(raw["gate"], g), _linear(raw["up"], g))
        return {"kind": kind, "layer": layer, "x": raw["x"]}
    if kind == "marlin":
        wm, sm = ops.repack_w4a16(raw["w"]["packed"], raw["w"]["scales"], g)
        return {"kind": kind, "words": wm, "scales": sm, "group": g, "x": raw["x"]}
    if kind == "packed":
        return {"kind": kind, "words": raw["w"]["packed"], "scales": raw["w"]["scales"].float(), "group": g,
                "x": raw["x"]}
    return {"kind": kind, "group": g, **raw["w"]}


def run(state: dict):
    kind = state["kind"]
    if kind == "stack":
        state["stack"].step()
        return state["stack"].outputs
    if kind in ("linear", "silu"):
        return state["layer"](state["x"])
    if kind == "marlin":
        return ops.gemm_w4a16_marlin(state["x"], state["words"], state["scales"], state["group"])
    if kind == "packed":
        return ops.gemm_w4a16(state["x"], state["words"], state["scales"], state["group"])
    if kind == "repack_gptq":
        return ops.repack_w4a16_gptq(state["qweight"], state["g_idx"], state["group"])
    return ops.repack_w4a16(state["packed"], state["scales"], state["group"])


# ---- what a pass cannot do without ------------------------------------------------------------


def _linear_work(m: int, k: int, n: int, case: dict, out: int, scale_bytes: int = 2) -> tuple[int, int]:
    kg = k // case["group"]
    b = k * n // 2 + kg * n * scale_bytes + 2 * m * (k + out)
    b += kg * n // 2 if case["zp"] else 0
    b += 4 * k if case["act"] else 0
    return b, 2 * m * k * n


def work(case: dict) -> dict:
    kind, m, k, n, g = case["kind"], case["m"], case["k"], case["n"], case["group"]
    if kind.startswith("repack"):
        words = (n + 63) // 64 * 64 * ((k + 63) // 64 * 64) // 2
        b = k * n // 2 + words
        b += (8 * k if case["act"] else 0) if kind == "repack_gptq" else 6 * (k // g) * n
        return {"bytes": b, "flops": 0}
    if kind == "stack":  # q|k|v, o, gate|up with its gate, down
        parts = [_linear_work(m, 4096, 6144, case, 6144), _linear_work(m, 4096, 4096, case, 4096),
                 _linear_work(m, k, 2 * n, case, n), _linear_work(m, n, k, case, k)]
        return {"bytes": case["layers"] * sum(p[0] for p in parts), "flops": case["layers"] * sum(p[1] for p in parts)}
    if kind == "silu":
        b, f = _linear_work(m, k, 2 * n, case, n)
    else:
        b, f = _linear_work(m, k, n, case, n, 2 if kind == "linear" else 4)
    return {"bytes": b, "flops": f}


# ---- results ----------------------------------------------------------------------------------


def tolerance(case: dict):
    """About four times the differences measured between the operators, the 64-bit result and the
    package's other kernels on the same inputs (relative, largest): fp16 outputs 2.1e-4 and 9e-4,
    their own rounding; bf16 outputs 3.2e-3 and 1.5e-2, where some kernels round the scaled
    weights to bf16 as the reference does; behind a SiLU gate, whose product scales each factor's
    error by the other, 4.5e-4 and 2.1e-3 in fp16, 4.7e-3 and 4.4e-2 in bf16."""
    if case["kind"].startswith("repack"):
        return "exact"
    gated = case["kind"] in ("silu", "stack")
    if case["dtype"] == "f16":
        return {"rel": 1.8e-3, "max": 8e-3} if gated else {"rel": 8e-4, "max": 3.6e-3}
    return {"rel": 1.8e-2, "max": 1.6e-1} if gated else {"rel": 1.2e-2, "max": 6e-2}


def _nibbles(words: torch.Tensor, dim: int) -> torch.Tensor:
    """The eight nibbles of each word along a new axis after `dim`, flattened into it."""
    parts = torch.stack([(words >> (4 * i)) & 0xF for i in range(8)], dim=dim + 1)
    return parts.flatten(dim, dim + 1)


def _dense_gptq(t: dict, group: int) -> torch.Tensor:
    """[K, N] in 64 bits: (u - z) * s by each row's group."""
    u = _nibbles(t["qweight"], 0)
    k, n = u.shape
    g = torch.arange(k, device=DEVICE) // group if t["g_idx"] is None else t["g_idx"].long()
    z = torch.full_like(t["scales"], 8, dtype=torch.int32) if t["qzeros"] is None else _nibbles(t["qzeros"], 1)
    return (u - z[g]).double() * t["scales"].double()[g]


def _dense_packed(t: dict, group: int) -> torch.Tensor:
    u = _nibbles(t["packed"], 1)
    q = torch.where(u >= 8, u - 16, u)
    return (q.double() * t["scales"].double().repeat_interleave(group, dim=1)).t()


def _silu_mul(g: torch.Tensor, u: torch.Tensor) -> torch.Tensor:
    return torch.nn.functional.silu(g) * u


def exact(case: dict, seed: int):
    kind, g = case["kind"], case["group"]
    if kind.startswith("repack"):
        return None  # whole words, compared as they are
    raw = _raw(case, seed)
    x = raw["x"].double()
    if kind == "stack":
        outs = []
        for t in raw["layers"]:
            def lin(name, v, t=t):
                return v @ _dense_gptq(t[name], g)
            h = _silu_mul(lin("gate", x), lin("up", x))
            outs += [torch.cat([lin("q", x), lin("k", x), lin("v", x)], dim=1), lin("o", x), h, lin("down", h)]
        return outs
    if kind == "silu":
        return _silu_mul(x @ _dense_gptq(raw["gate"], g), x @ _dense_gptq(raw["up"], g))
    return x @ (_dense_gptq(raw["w"], g) if kind == "linear" else _dense_packed(raw["w"], g))
