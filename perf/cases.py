"""What a program built on this package has it do, as cases that can be timed and compared:
EXL3 linears on their own, the linears and glue of a dense decoder layer, and MoE layers,
from one decoded token to a long prompt.

`listed()` names the cases, `draw(rng)` gives another one of the same ranges, `prepare` builds
the weights and inputs such a program holds, `run` is one pass through the public classes of
`berth_amd.device` and `berth_amd.moe`.
"""
import math

import numpy as np
import torch

from berth_amd import kernels as K
from berth_amd import synth
from berth_amd.device import Exl3Linear, Exl3MultiLinear, Gpu, MlpLayer, RowScratch
from berth_amd.kernels import Codebook, OutDtype
from berth_amd.moe import MoeLayer

CODEBOOKS = {"3inst": Codebook.DEFAULT, "mcg": Codebook.MCG, "mul1": Codebook.MUL1}
FORWARD_N_ROWS = 144        # Exl3Linear.forward_n takes up to this many rows, forward_rows more


def _linear(name, rows, k, n, bits, codebook="mul1", out="f16"):
    return {"name": name, "kind": "linear", "rows": rows, "k": k, "n": n, "bits": bits, "codebook": codebook, "out": out}


def _layer(name, rows, bits=4, codebook="mul1", hidden=5120, q=6144, kv=1024, inter=17408):
    return {"name": name, "kind": "layer", "rows": rows, "hidden": hidden, "q": q, "kv": kv, "inter": inter,
            "bits": bits, "codebook": codebook}


def _moe(name, rows, hidden=2048, experts=128, top_k=8, inter=768, bits=4, shared=False, zipf=False):
    return {"name": name, "kind": "moe", "rows": rows, "hidden": hidden, "experts": experts, "top_k": top_k,
            "inter": inter, "bits": bits, "codebook": "mul1", "shared": shared, "zipf": zipf}


def listed():
    return [
        # one square linear, one token: the smallest call a decoding program makes, where latency counts
        _linear("linear_1x4096x4096", 1, 4096, 4096, 4),
        # one token, odd multiples of 128, the reference's older codebook, fp32 out (a residual-stream linear)
        _linear("linear_1x2688x7296_5bpw", 1, 2688, 7296, 5, "mcg", "f32"),
        # the output head of a 27B-shaped model for one token
        _linear("lm_head_1x5120x248320_6bpw", 1, 5120, 248320, 6),
        # one decoder layer of a 27B-shaped model while decoding: the step a user waits for, layer after layer
        _layer("layer_decode_1", 1),
        # the same layer on a handful of rows: checking drafted tokens, or a few requests at a time
        _layer("layer_verify_5_3bpw", 5, bits=3, codebook="mcg"),
        # a small batch, or the last rows of a prompt
        _layer("layer_batch_24", 24),
        # a 100-token prompt
        _layer("layer_prompt_100", 100),
        # a 1500-token prompt: the largest dense case
        _layer("layer_prompt_1500", 1500),
        # one token through an A3B-style MoE layer
        _moe("moe_decode_1", 1),
        # 64 requests decoding together
        _moe("moe_batch_64", 64),
        # many small experts, an always-on one, and a few experts that most tokens choose
        _moe("moe_skewed_256_3bpw", 256, experts=512, top_k=10, inter=512, bits=3, shared=True, zipf=True),
        # a 1500-token prompt through the A3B-style layer
        _moe("moe_prompt_1500", 1500),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _blocks(rng, lo, hi):
    """A multiple of 128 (one Hadamard block) between lo and hi."""
    return 128 * _log_uniform(rng, lo // 128, hi // 128)


def draw(rng):
    codebook = rng.choice(["mul1", "mul1", "mul1", "mcg", "3inst"])
    kind = rng.choice(["linear", "layer", "layer", "moe"])
    decode = rng.random() < 0.35
    if kind == "linear":
        k, n = _blocks(rng, 1024, 17408), _blocks(rng, 1024, 32768)
        rows = min(_log_uniform(rng, 2, 1500), 500_000_000_000 // (k * n))      # no larger than the largest listed case
        case = _linear("", 1 if decode else rows, k, n, rng.choice([2, 3, 4, 5, 6]), codebook, rng.choice(["f16", "f32"]))
    elif kind == "layer":
        hidden = _blocks(rng, 1024, 5120)
        kv = 128 * rng.choice([2, 4, 8])
        q = kv * rng.randint(1, max(1, min(6144, int(1.5 * hidden)) // kv))
        inter = min(17408, 128 * int(hidden * rng.uniform(2.0, 3.6) / 128))
        case = _layer("", 1 if decode else _log_uniform(rng, 2, 1500), rng.choice([2, 3, 4, 5]), codebook,
                      hidden, q, kv, inter)
    else:
        experts = rng.choice([16, 32, 60, 64, 128, 256, 512])
        skewed = rng.random() < 0.4
        case = _moe("", 1 if decode else _log_uniform(rng, 2, 1500), _blocks(rng, 1024, 2048), experts,
                    rng.choice([4, 6, 8, 10]), _blocks(rng, 512, 1024), rng.choice([3, 4]), rng.random() < 0.5, skewed)
    del case["name"]
    return case


# ---- what a program holds before it calls -----------------------------------------------------

_GPU = None


def _gpu():
    global _GPU
    if _GPU is None:
        _GPU = Gpu()
    return _GPU


class _Source:
    """Seeded tensors made on the device, in the distributions of `berth_amd.synth`."""

    def __init__(self, seed):
        self.device = _gpu().device
        self.g = torch.Generator(device=self.device)
        self.g.manual_seed(seed)

    def words(self, *shape):
        return torch.randint(-32768, 32768, shape, dtype=torch.int16, device=self.device, generator=self.g)

    def scales(self, *shape):
        sign = torch.randint(0, 2, shape, device=self.device, generator=self.g).float() * 2 - 1
        return (sign * torch.exp(0.1 * torch.randn(shape, device=self.device, generator=self.g))).half()

    def normal(self, shape, dtype, sigma=1.0):
        return (sigma * torch.randn(shape, device=self.device, generator=self.g)).to(dtype)

    def empty(self, *shape, dtype=torch.float16):
        return torch.zeros(shape, dtype=dtype, device=self.device)

    def linear(self, name, k, n, bits, codebook):
        return Exl3Linear.from_device(name, self.words(k * n * bits // 16), self.scales(k), self.scales(n), bits, codebook)


def _prepare_linear(case, src):
    rows, k, n = case["rows"], case["k"], case["n"]
    out = OutDtype.F32 if case["out"] == "f32" else OutDtype.F16
    return {"linear": src.linear("linear", k, n, case["bits"], CODEBOOKS[case["codebook"]]), "rows": rows, "out": out,
            "a": src.normal((rows, k), torch.float16),
            "c": src.empty(rows, n, dtype=torch.float32 if case["out"] == "f32" else torch.float16),
            "a_had": src.empty(rows, k) if 1 < rows <= FORWARD_N_ROWS else None,
            "scratch": RowScratch(_gpu(), rows, k, n) if rows > FORWARD_N_ROWS else None}


def _prepare_layer(case, src):
    gpu, rows, hidden, q, kv, inter = _gpu(), case["rows"], case["hidden"], case["q"], case["kv"], case["inter"]
    bits, codebook = case["bits"], CODEBOOKS[case["codebook"]]
    qkv = Exl3MultiLinear(gpu, [src.linear(name, hidden, n, bits, codebook)
                                for name, n in (("q_proj", q), ("k_proj", kv), ("v_proj", kv))])
    mlp = MlpLayer(gpu, src.linear("gate_proj", hidden, inter, bits, codebook),
                   src.linear("up_proj", hidden, inter, bits, codebook),
                   src.linear("down_proj", inter, hidden, bits, codebook), max_rows=rows)
    f32 = torch.float32
    return {"qkv": qkv, "o": src.linear("o_proj", q, hidden, bits, codebook), "mlp": mlp, "rows": rows, "hidden": hidden,
            # the residual stream, the norm weights (stored as an offset from one) and what attention hands over
            "residual": src.normal((rows, hidden), f32), "norm_1": src.normal((hidden,), torch.bfloat16, 0.1),
            "norm_2": src.normal((hidden,), torch.bfloat16, 0.1), "attended": src.normal((rows, q), torch.float16),
            "h": src.empty(rows, hidden), "q": src.empty(rows, q), "k": src.empty(rows, kv), "v": src.empty(rows, kv),
            "o_out": src.empty(rows, hidden, dtype=f32), "residual_out": src.empty(rows, hidden, dtype=f32),
            "y": src.empty(rows, hidden, dtype=f32),
            "a_had": src.empty(rows, q) if 1 < rows <= FORWARD_N_ROWS else None,
            "scratch": RowScratch(gpu, rows, q, hidden) if rows > FORWARD_N_ROWS else None}


def _prepare_moe(case, src, seed):
    gpu, rows, hidden, E, inter = _gpu(), case["rows"], case["hidden"], case["experts"], case["inter"]
    bits, codebook, n = case["bits"], CODEBOOKS[case["codebook"]], case["experts"] + (1 if case["shared"] else 0)
    words = src.words(n, 3, hidden * inter * bits // 16)
    wide, narrow = src.scales(n, 3, hidden), src.scales(n, 3, inter)
    a_had = src.empty(max(hidden, inter))
    experts = [tuple(Exl3Linear.from_device(name, words[e, j], (wide, narrow)[j == 2][e, j], (narrow, wide)[j == 2][e, j],
                                            bits, codebook, a_had)
                     for j, name in enumerate(("gate_proj", "up_proj", "down_proj"))) for e in range(n)]
    layer = MoeLayer(gpu, synth.router_weight(seed, hidden, E), experts[:E], case["top_k"],
                     shared=experts[E] if case["shared"] else None, bias=synth.zipf_bias(seed, E) if case["zipf"] else None,
                     codebook=codebook)
    return {"layer": layer, "rows": rows, "x": src.normal((rows, hidden), torch.float16),
            "out": src.empty(rows, hidden, dtype=torch.float32),
            "idx": src.empty(rows, case["top_k"], dtype=torch.int32), "w": src.empty(rows, case["top_k"], dtype=torch.float32)}


def prepare(case, seed):
    src = _Source(seed)
    if case["kind"] == "linear":
        state = _prepare_linear(case, src)
    elif case["kind"] == "layer":
        state = _prepare_layer(case, src)
    else:
        state = _prepare_moe(case, src, seed)
    state["kind"] = case["kind"]
    return state


# ---- one pass ---------------------------------------------------------------------------------

def _forward(gpu, linear, a, c, rows, out, a_had, scratch):
    if rows == 1:
        linear.forward(gpu, a, c, out)
    elif rows <= FORWARD_N_ROWS:
        linear.forward_n(gpu, a_had, a, c, rows, out)
    else:
        linear.forward_rows(gpu, scratch, a, c, rows, out)


def run(state):
    gpu, rows = _gpu(), state["rows"]
    if state["kind"] == "linear":
        _forward(gpu, state["linear"], state["a"], state["c"], rows, state["out"], state["a_had"], state["scratch"])
        return state["c"]
    if state["kind"] == "moe":
        state["layer"].forward(gpu, state["x"], state["out"], rows, state["idx"], state["w"])
        return {"out": state["out"], "idx": state["idx"], "w": state["w"]}
    # a decoder layer without attention itself: norm, q / k / v, the output projection of what
    # attention returned, then the block residual add - norm - MLP - residual add
    K.ops.rms_norm(state["residual"].data_ptr(), state["norm_1"].data_ptr(), state["h"].data_ptr(), rows, state["hidden"],
                   1e-6, stream=gpu.raw_stream())
    state["qkv"].forward(gpu, state["h"], [state["q"], state["k"], state["v"]], OutDtype.F16, rows)
    _forward(gpu, state["o"], state["attended"], state["o_out"], rows, OutDtype.F32, state["a_had"], state["scratch"])
    state["mlp"].forward_block(gpu, state["o_out"], state["residual"], state["residual_out"], state["norm_2"], state["y"],
                               rows=rows)
    return {name: state[name] for name in ("q", "k", "v", "o_out", "residual_out", "y")}


# ---- what a pass cannot do without ------------------------------------------------------------

def _linear_work(rows, k, n, bits, out_bytes, in_bytes=2):
    """Weights and scales once, the input read, the output written."""
    return k * n * bits / 8 + 2 * k + 2 * n + in_bytes * rows * k + out_bytes * rows * n, 2.0 * rows * k * n


def _experts_hit(case):
    """Distinct experts that the tokens choose, from router logits of the spread the inputs give."""
    rng = np.random.default_rng(5)
    E, k = case["experts"], case["top_k"]
    logits = rng.normal(0.0, 0.02 * math.sqrt(case["hidden"]), size=(case["rows"], E))
    if case["zipf"]:
        logits -= 1.1 * np.log(rng.permutation(E) + 1.0)
    return len(np.unique(np.argpartition(-logits, k - 1, axis=1)[:, :k]))


def work(case):
    rows, bits = case["rows"], case["bits"]
    if case["kind"] == "linear":
        nbytes, flops = _linear_work(rows, case["k"], case["n"], bits, 4 if case["out"] == "f32" else 2)
    elif case["kind"] == "layer":
        hidden, q, kv, inter = case["hidden"], case["q"], case["kv"], case["inter"]
        # q / k / v write fp16; the activations between the launches need not reach memory
        parts = [_linear_work(rows, hidden, q + 2 * kv, bits, 2, 0), _linear_work(rows, q, hidden, bits, 4),
                 _linear_work(rows, hidden, 2 * inter, bits, 0, 0), _linear_work(rows, inter, hidden, bits, 4, 0)]
        nbytes = sum(p[0] for p in parts) + 4 * rows * hidden * 2 + 2 * 2 * hidden     # residual in and out, norm weights
        flops = sum(p[1] for p in parts)
    else:
        hidden, inter, E, k = case["hidden"], case["inter"], case["experts"], case["top_k"]
        expert = 3 * hidden * inter * bits / 8 + 2 * 3 * (hidden + inter)
        n = _experts_hit(case) + (1 if case["shared"] else 0)
        nbytes = n * expert + 2 * hidden * E + rows * (2 * hidden + 4 * hidden + 8 * k)
        flops = 2.0 * rows * hidden * E + 2.0 * rows * (k + (1 if case["shared"] else 0)) * 3 * hidden * inter
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    # fp16 activations and weights, products summed in fp32: half a unit in the last place of
    # fp16 is 4.9e-4 of a value; chosen experts are whole numbers and stay the same
    return {"rel": 1e-3}
