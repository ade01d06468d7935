"""Timed workloads of the gated-mixture framework, from one decode call to a
whole decoder training step, each through its public entry points.

A case is a dict of plain values; its "kind" picks the path:

  linear     MixedQuantLinear, forward and backward (gradients of the input
             and the gates), or the forward alone ("grad": False)
  routed     the per-token routed forward of a gated Linear and its backward
  mlp        one SwiGLU block of gated Linears, forward and backward
  embedding  MixedQuantEmbedding lookup, forward and backward
  attention  rotary embedding + causal attention, forward and backward
  loss       CE + KL distillation loss and the gradient of the logits
  dequant    fp32 decode of one packed tensor per candidate format
  step       the 0.8B-class decoder's gate-training step (GateTrainer.step)

Candidates are random valid GGUF blocks whose scales give weights of a few
hundredths, as a decoder's are; activations and gradients are N(0, 1) bf16,
gate logits N(0, 1).
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "voodoo-dyn-quant_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from voodoo_quant import _hip, layers  # noqa: E402
from voodoo_quant.training import step as training_step  # noqa: E402
from voodoo_quant.training import trainer  # noqa: E402

DEV = "cuda"
K6 = "Q2_K,Q3_K,Q4_K,Q5_K,Q6_K,Q8_0"
K4 = "Q3_K,Q4_K,Q6_K,Q8_0"
K8 = "Q2_K,IQ2_XXS,Q3_K,IQ3_S,Q4_K,Q5_K,Q6_K,Q8_0"       # the wide stress menu
RECIPE = "Q8_0,Q5_K,IQ3_S,IQ2_S,IQ2_XXS,IQ1_S"           # a low-bit recipe's menu

GGML_IDS = {"Q8_0": 8, "Q2_K": 10, "Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "IQ2_XXS": 16, "IQ1_S": 19,
            "IQ3_S": 21, "IQ2_S": 22}
# bytes per 256 weights, and the offsets and smallest values of the fp16 scale
# fields: (offset within a block, base); Q8_0 has eight 34-byte blocks.  The
# bases keep decoded weights within about +-0.2.
GROUP_BYTES = {"Q8_0": 272, "Q2_K": 84, "Q3_K": 110, "Q4_K": 144, "Q5_K": 176, "Q6_K": 210, "IQ2_XXS": 66,
               "IQ1_S": 50, "IQ3_S": 110, "IQ2_S": 82}
SCALES = {"Q8_0": ((0, 2.0 ** -11),), "Q2_K": ((80, 2.0 ** -9), (82, 1.5 * 2.0 ** -9)), "Q3_K": ((108, 2.0 ** -11),),
          "Q4_K": ((0, 2.0 ** -14), (2, 7.5 * 2.0 ** -14)), "Q5_K": ((0, 2.0 ** -15), (2, 15.5 * 2.0 ** -15)),
          "Q6_K": ((208, 2.0 ** -16),), "IQ1_S": ((0, 2.0 ** -8),), "IQ2_XXS": ((0, 2.0 ** -11),),
          "IQ2_S": ((0, 2.0 ** -11),), "IQ3_S": ((0, 2.0 ** -13),)}


def listed():
    return [
        # the smallest layer call: a 1024-wide projection on one short batch, four candidates
        {"name": "linear_512x1024x1024_k4", "kind": "linear", "tokens": 512, "d": 1024, "n": 1024, "types": K4,
         "grad": True},
        # evaluation with the gates still soft: one sequence's next token through a 27B-class MLP projection
        {"name": "linear_eval_1x5120x17408", "kind": "linear", "tokens": 1, "d": 5120, "n": 17408, "types": K6,
         "grad": False},
        # gate training on a short prompt: a 27B-class attention projection, an odd token count
        {"name": "linear_61x5120x6144", "kind": "linear", "tokens": 61, "d": 5120, "n": 6144, "types": K6,
         "grad": True},
        # a ragged mid-size batch through the stress stack's projection, code-book formats in the menu
        {"name": "linear_1000x4096x14336_k8", "kind": "linear", "tokens": 1000, "d": 4096, "n": 14336, "types": K8,
         "grad": True},
        # the headline layer: a 27B-class MLP projection at a full training batch
        {"name": "linear_8192x5120x17408", "kind": "linear", "tokens": 8192, "d": 5120, "n": 17408, "types": K6,
         "grad": True},
        # per-token routing through the same class of projection
        {"name": "routed_4096x5120x6144", "kind": "routed", "tokens": 4096, "d": 5120, "n": 6144, "types": K6},
        # one MLP block of the 0.8B-class decoder at its training batch
        {"name": "mlp_8192x1024x3072", "kind": "mlp", "tokens": 8192, "hidden": 1024, "mlp": 3072, "types": K6},
        # the token embedding of that decoder: vocabulary-sized candidates, one batch of ids
        {"name": "embedding_8192x1024", "kind": "embedding", "ids": 8192, "vocab": 151936, "dim": 1024, "types": K6},
        # its attention: 4 sequences of 2048 positions, grouped K/V heads
        {"name": "attention_4x2048_h16_kv4", "kind": "attention", "batch": 4, "seq": 2048, "heads": 16,
         "kv_heads": 4},
        # its distillation loss over a quarter batch of logits, softened
        {"name": "loss_2048x151936", "kind": "loss", "rows": 2048, "vocab": 151936, "temperature": 2.0},
        # decoding a tensor's candidates to fp32 for export and inspection
        {"name": "dequant_4096x14336", "kind": "dequant", "rows": 4096, "cols": 14336, "types": K6},
        # the whole training step as a trainer runs it
        {"name": "step_0p8b_4x2048", "kind": "step", "batch": 4, "seq": 2048, "layers": 24},
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, int(v) // multiple * multiple)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "routed", "mlp", "embedding", "attention", "loss",
                       "dequant"])
    types = rng.choice([K6, K6, K4, K8, RECIPE])
    if kind in ("linear", "routed"):
        # widths from a 1024-wide decoder to a 27B-class one; a third of them off the 256-weight grid
        m8 = rng.choice([256, 256, 8])
        d, n = _log_int(rng, 1024, 17408, m8), _log_int(rng, 1024, 17408, m8)
        while d * n > 5120 * 17408:
            d, n = _log_int(rng, 1024, 17408, m8), _log_int(rng, 1024, 17408, m8)
        if kind == "routed":
            return {"kind": kind, "tokens": _log_int(rng, 256, 8192), "d": d, "n": n, "types": types}
        return {"kind": kind, "tokens": _log_int(rng, 1, 8192), "d": d, "n": n, "types": types,
                "grad": rng.random() < 0.8}
    if kind == "mlp":
        return {"kind": kind, "tokens": _log_int(rng, 64, 8192), "hidden": _log_int(rng, 1024, 4096, 256),
                "mlp": _log_int(rng, 2048, 8192, 256), "types": types}
    if kind == "embedding":
        return {"kind": kind, "ids": _log_int(rng, 1, 16384), "vocab": _log_int(rng, 32000, 151936),
                "dim": _log_int(rng, 1024, 5120, rng.choice([256, 8])), "types": types}
    if kind == "attention":
        kv = rng.choice([1, 2, 4, 8])
        return {"kind": kind, "batch": rng.randint(1, 4), "seq": _log_int(rng, 64, 2048),
                "heads": kv * rng.choice([1, 2, 4]), "kv_heads": kv}
    if kind == "loss":
        return {"kind": kind, "rows": _log_int(rng, 16, 2048), "vocab": _log_int(rng, 32000, 151936, 8),
                "temperature": rng.choice([1.0, 2.0])}
    return {"kind": kind, "rows": _log_int(rng, 256, 4096), "cols": _log_int(rng, 1024, 14336, 256), "types": types}


# ---------------------------------------------------------------- inputs
def _pad256(d):
    return (d + 255) // 256 * 256


def _packed(qt, rows, cols, gen):
    """Random valid blocks of an [rows, cols] tensor, rows padded to 256 weights."""
    blocks = rows * _pad256(cols) // (32 if qt == "Q8_0" else 256)
    size = 34 if qt == "Q8_0" else GROUP_BYTES[qt]
    q = torch.randint(0, 256, (blocks, size), dtype=torch.uint8, device=DEV, generator=gen)
    for off, base in SCALES[qt]:
        h = (base * (1.0 + torch.rand(blocks, device=DEV, generator=gen))).to(torch.float16)
        q[:, off:off + 2] = h.view(torch.uint8).view(blocks, 2)
    return q.reshape(-1)


def _bf16(gen, *shape):
    return torch.randn(*shape, device=DEV, generator=gen).to(torch.bfloat16)


def _gates(gen, k):
    return torch.randn(k, device=DEV, generator=gen)


def _inputs(case, seed):
    """The case's plain tensors: what both the framework and a reference read."""
    gen = torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + 17)
    kind = case["kind"]
    types = case.get("types", K6).split(",")
    if kind in ("linear", "routed"):
        s = {"qbytes": [_packed(t, case["n"], case["d"], gen) for t in types], "gates": _gates(gen, len(types)),
             "x": _bf16(gen, case["tokens"], case["d"])}
        if kind == "routed" or case["grad"]:
            s["dy"] = _bf16(gen, case["tokens"], case["n"])
        if kind == "routed":
            p = torch.softmax(s["gates"], 0)
            s["routing"] = torch.multinomial(p, case["tokens"], replacement=True, generator=gen)
        return s
    if kind == "mlp":
        h, m = case["hidden"], case["mlp"]
        return {"tensors": {name: ([_packed(t, o, i, gen) for t in types], _gates(gen, len(types)))
                            for name, (o, i) in (("gate", (m, h)), ("up", (m, h)), ("down", (h, m)))},
                "x": _bf16(gen, case["tokens"], h), "dy": _bf16(gen, case["tokens"], h)}
    if kind == "embedding":
        return {"qbytes": [_packed(t, case["vocab"], case["dim"], gen) for t in types],
                "gates": _gates(gen, len(types)),
                "ids": torch.randint(0, case["vocab"], (case["ids"],), device=DEV, generator=gen),
                "dy": _bf16(gen, case["ids"], case["dim"])}
    if kind == "attention":
        b, s, hq, hk = case["batch"], case["seq"], case["heads"], case["kv_heads"]
        inv = 1.0 / (1.0e6 ** (torch.arange(0, 64, 2, dtype=torch.float64, device=DEV) / 64))
        ang = torch.outer(torch.arange(s, dtype=torch.float64, device=DEV), inv)
        ang = torch.cat([ang, ang], dim=-1)
        return {"qkv": _bf16(gen, b * s, (hq + 2 * hk) * 64), "dout": _bf16(gen, b, s, hq, 64),
                "cos": ang.cos().float().contiguous(), "sin": ang.sin().float().contiguous()}
    if kind == "loss":
        r, v = case["rows"], case["vocab"]
        t = 2.0 * torch.randn(r, v, device=DEV, generator=gen)
        logits = (t + torch.randn(r, v, device=DEV, generator=gen)).to(torch.bfloat16)
        labels = torch.randint(0, v, (r,), device=DEV, generator=gen)
        labels[torch.rand(r, device=DEV, generator=gen) < 0.02] = -100  # ignored positions
        labels[0] = 1
        return {"logits": logits, "teacher": t.to(torch.bfloat16), "labels": labels}
    if kind == "dequant":
        return {"qbytes": [_packed(t, case["rows"], case["cols"], gen) for t in types]}
    raise ValueError(kind)


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "step":
        cfg = training_step.DecoderConfig(layers=case["layers"])
        student, teacher, replaced = training_step.build_models(cfg, K6.split(","), DEV, seed=int(seed))
        # the settings the benchmark trains with
        state["trainer"] = training_step.GateTrainer(
            student, teacher, replaced,
            training_step.StepConfig(max_steps=1000, teacher_stream=True, tuned_gemms=True),
            total_8bit_bytes=float(cfg.gated_weights()))
        gen = torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + 17)
        for p in state["trainer"].trainable:
            p.data.copy_(0.5 * torch.randn(p.shape, device=DEV, generator=gen))
        ids = torch.randint(0, cfg.vocab, (case["batch"], case["seq"] + 1), device=DEV, generator=gen)
        state["x"], state["y"] = ids[:, :-1].contiguous(), ids[:, 1:].contiguous()
        return state
    data = _inputs(case, seed)
    types = case.get("types", K6).split(",")
    if kind in ("linear", "routed"):
        if kind == "routed":  # the bf16 decodes a routed layer keeps while its candidates stay fixed
            d_pad = _pad256(case["d"])
            data["decoded"] = [_hip.dequant_bf16(GGML_IDS[t], q, case["n"], d_pad)
                               for t, q in zip(types, data["qbytes"])]
            data["meta"] = (tuple(GGML_IDS[t] for t in types), case["n"], d_pad)
            data["gates"].requires_grad_(True)
        else:
            data["module"] = layers.MixedQuantLinear.from_packed(case["d"], case["n"], types, data.pop("qbytes"))
            data["module"].gates.data.copy_(data.pop("gates"))
        if kind == "routed" or case["grad"]:
            data["x"].requires_grad_(True)
    elif kind == "mlp":
        mods = {}
        for name, (qbytes, gates) in data.pop("tensors").items():
            o, i = (case["hidden"], case["mlp"]) if name == "down" else (case["mlp"], case["hidden"])
            mods[f"mlp.{name}_proj"] = layers.MixedQuantLinear.from_packed(i, o, types, qbytes)
            mods[f"mlp.{name}_proj"].gates.data.copy_(gates)
        cfg = training_step.StackConfig(blocks=1, hidden=case["hidden"], mlp=case["mlp"])
        data["stack"] = training_step.SwiGLUStack(cfg, [mods], torch.device(DEV))
        data["gates"] = [mods[f"mlp.{n}_proj"].gates for n in ("gate", "up", "down")]
        data["x"].requires_grad_(True)
    elif kind == "embedding":
        mod = layers.MixedQuantEmbedding.from_packed(case["vocab"], case["dim"], types, data.pop("qbytes"))
        mod.gates.data.copy_(data.pop("gates"))
        mod.id_check = "deferred"  # as the trainer sets it
        data["module"] = mod
    elif kind == "loss":
        data["logits"].requires_grad_(True)
    state.update(data)
    return state


# ---------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        mod, x = state["module"], state["x"]
        if not case["grad"]:
            with torch.no_grad():
                return {"y": mod(x)}
        y = mod(x)
        dx, dgates = torch.autograd.grad(y, (x, mod.gates), state["dy"])
        return {"y": y.detach(), "dx": dx, "dgates": dgates}
    if kind == "routed":
        x, gates = state["x"], state["gates"]
        y = layers.RoutedLinearFunction.apply(x, torch.softmax(gates, 0), state["routing"], state["meta"],
                                              state["decoded"], *state["qbytes"])
        dx, dgates = torch.autograd.grad(y, (x, gates), state["dy"])
        return {"y": y.detach(), "dx": dx, "dgates": dgates}
    if kind == "mlp":
        y = state["stack"](state["x"])
        grads = torch.autograd.grad(y, [state["x"], *state["gates"]], state["dy"])
        return {"y": y.detach(), "dx": grads[0], "dgates": list(grads[1:])}
    if kind == "embedding":
        layers.raise_pending_id_errors(block=False)
        mod = state["module"]
        y = mod(state["ids"])
        (dgates,) = torch.autograd.grad(y, (mod.gates,), state["dy"])
        return {"y": y.detach(), "dgates": dgates}
    if kind == "attention":
        b, s, hq, hk = case["batch"], case["seq"], case["heads"], case["kv_heads"]
        cos, sin = state["cos"], state["sin"]
        q, k, v = _hip.rope_qkv_fwd(state["qkv"], b, s, hq, hk, 64, cos, sin, repeat_kv=False)
        q, k, v = (t.view(b, s, -1, 64).transpose(1, 2) for t in (q, k, v))
        out, lse = _hip.attention_fwd(q, k, v)
        dq, dk, dv = _hip.attention_bwd(state["dout"].transpose(1, 2), q, k, v, out, lse)
        return {"out": out, "dqkv": _hip.rope_qkv_bwd(dq, dk, dv, b, s, hq, hk, 64, cos, sin)}
    if kind == "loss":
        ce, kl = trainer.distill_losses_fused(state["logits"], state["teacher"], state["labels"],
                                              case["temperature"])
        (g,) = torch.autograd.grad(ce + kl, (state["logits"],))
        return {"ce": ce.detach(), "kl": kl.detach(), "dlogits": g}
    if kind == "dequant":
        return [layers.dequantize_tensor_gpu_fp32(q, t, case["rows"], case["cols"], q.device)
                for q, t in zip(state["qbytes"], case["types"].split(","))]
    tr = state["trainer"]
    losses = tr.step(state["x"], state["y"])
    # the optimizer's first moments: the clipped gate gradients, averaged
    moments = [tr.opt.state[p]["exp_avg"] for p in tr.trainable]
    return {"lm": losses["lm"], "kl": losses["kl"], "size": losses["size"], "moments": moments}


# ---------------------------------------------------------------- what a pass cannot do without
def _packed_bytes(case, rows, cols):
    return sum(rows * (_pad256(cols) // 256) * GROUP_BYTES[t] for t in case["types"].split(","))


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, d, n = case["tokens"], case["d"], case["n"]
        packed = _packed_bytes(case, n, d)
        if not case["grad"]:
            return {"bytes": packed + 2 * m * (d + n), "flops": 2 * m * n * d}
        # forward and backward each need the candidates, X, and Y or dY; the backward writes dX
        return {"bytes": 2 * packed + 2 * m * (3 * d + 2 * n), "flops": 6 * m * n * d}
    if kind == "routed":
        m, d, n = case["tokens"], case["d"], case["n"]
        k = len(case["types"].split(","))
        # the forward reads the kept bf16 decodes
        return {"bytes": 2 * k * n * d + _packed_bytes(case, n, d) + 2 * m * (3 * d + 2 * n), "flops": 6 * m * n * d}
    if kind == "mlp":
        m, h, f = case["tokens"], case["hidden"], case["mlp"]
        packed = 2 * _packed_bytes(case, f, h) + _packed_bytes(case, h, f)
        return {"bytes": 2 * packed + 2 * m * 4 * h, "flops": 18 * m * h * f}
    if kind == "embedding":
        row = _packed_bytes(case, 1, case["dim"])
        return {"bytes": case["ids"] * (2 * row + 4 * case["dim"] + 16), "flops": 0}
    if kind == "attention":
        b, s, hq, hk = case["batch"], case["seq"], case["heads"], case["kv_heads"]
        pairs = b * hq * s * (s + 1) // 2
        # two products forward, five backward, over the visible pairs; qkv read twice, dout and out read,
        # out and dqkv written
        return {"bytes": 2 * b * s * 64 * (3 * (hq + 2 * hk) + 3 * hq), "flops": 7 * 2 * 64 * pairs}
    if kind == "loss":
        return {"bytes": 10 * case["rows"] * case["vocab"], "flops": 0}
    if kind == "dequant":
        types = case["types"].split(",")
        return {"bytes": _packed_bytes(case, case["rows"], case["cols"]) + 4 * case["rows"] * case["cols"] * len(types),
                "flops": 0}
    cfg = training_step.DecoderConfig(layers=case["layers"])
    tokens = case["batch"] * case["seq"]
    weights = cfg.layers * sum(o * i for o, i in cfg.linear_shapes().values())
    per_weight = sum(GROUP_BYTES[t] for t in K6.split(",")) / 256.0
    # candidates twice, the teacher's bf16 weights and both heads, logits of both models and their gradient
    nbytes = 2 * per_weight * weights + 2 * weights + 6 * cfg.vocab * cfg.hidden + 10 * tokens * cfg.vocab
    return {"bytes": int(nbytes), "flops": int(training_step.step_flops(cfg, tokens, case["seq"]))}


# ---------------------------------------------------------------- tolerances
def tolerance(case):
    # about four times the largest distance to exact() seen over the listed cases and 14 drawn ones
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "step":
        # seen: 5e-4 and 7e-3 between the step and itself with torch's attention, single projections, or
        # the decoder's glue as torch operations
        return {"rel": 2e-3, "max": 3e-2}
    if kind == "mlp":
        # gate gradients: sums whose terms, from bf16 activations, cancel to a hundredth (seen 1.1e-2)
        return {"rel": 3e-2, "max": 0.1}
    if kind == "attention":
        # probabilities and score gradients in bf16 (seen 3.7e-3 and 0.15)
        return {"rel": 1.5e-2, "max": 0.6}
    if kind == "loss":
        # one bf16 rounding of the gradient (seen 3.7e-3 and 3.9e-3)
        return {"rel": 1.5e-2, "max": 1.6e-2}
    if kind == "embedding":
        # one bf16 rounding of a row (seen 1.7e-3 and 3.9e-3)
        return {"rel": 7e-3, "max": 1.6e-2}
    # linear, routed: bf16 rounding of the mixed weight and of the output (seen 2.4e-3 and 1.4e-2)
    return {"rel": 1e-2, "max": 5e-2}


# ---------------------------------------------------------------- 64-bit references
def _decode64(qt, q, rows, cols):
    """float64 [rows, cols padded to 256] weights of packed blocks, from the public GGUF block layouts; None
    for the formats that need code books of thousands of entries."""
    if qt.startswith("IQ"):
        return None
    size = 34 if qt == "Q8_0" else GROUP_BYTES[qt]
    b = q.view(-1, size)
    nb = b.shape[0]

    def f16(off):
        return b[:, off:off + 2].contiguous().view(torch.float16).double().view(nb, 1)

    def i32(t):
        return t.to(torch.int32)

    if qt == "Q8_0":
        w = f16(0) * b[:, 2:34].contiguous().view(torch.int8).double()
    elif qt in ("Q4_K", "Q5_K"):
        s = i32(b[:, 4:16])
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = i32(b[:, (48 if qt == "Q5_K" else 16):]).view(nb, 4, 1, 32)
        v = torch.cat([qs & 15, qs >> 4], 2).view(nb, 8, 32)
        if qt == "Q5_K":
            hi = i32(b[:, 16:48]).view(nb, 1, 32)
            sh = torch.arange(8, device=q.device, dtype=torch.int32).view(1, 8, 1)
            v = v + (((hi >> sh) & 1) << 4)
        w = f16(0).view(nb, 1, 1) * sc.double().view(nb, 8, 1) * v - f16(2).view(nb, 1, 1) * mn.double().view(nb, 8, 1)
    elif qt == "Q6_K":
        ql = i32(b[:, :128]).view(nb, 2, 2, 32)
        qh = i32(b[:, 128:192]).view(nb, 2, 1, 32)
        sh = torch.tensor([0, 2, 4, 6], device=q.device, dtype=torch.int32).view(1, 1, 4, 1)
        v = (torch.cat([ql & 15, ql >> 4], 2) | (((qh >> sh) & 3) << 4)) - 32   # [nb, 2, 4, 32]
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(nb, 2, 4, 2, 1)
        w = f16(208).view(nb, 1, 1, 1, 1) * sc * v.view(nb, 2, 4, 2, 16)
    else:
        sh = torch.tensor([0, 2, 4, 6], device=q.device, dtype=torch.int32).view(1, 1, 4, 1)
        if qt == "Q2_K":
            v = (i32(b[:, 16:80]).view(nb, 2, 1, 32) >> sh) & 3
            s = i32(b[:, :16]).view(nb, 2, 4, 2, 1)
            w = (f16(80).view(nb, 1, 1, 1, 1) * (s & 15) * v.view(nb, 2, 4, 2, 16)
                 - f16(82).view(nb, 1, 1, 1, 1) * (s >> 4))
        else:  # Q3_K
            v = (i32(b[:, 32:96]).view(nb, 2, 1, 32) >> sh) & 3
            bit = torch.arange(8, device=q.device, dtype=torch.int32).view(1, 2, 4, 1)
            v = v - 4 * (1 - ((i32(b[:, :32]).view(nb, 1, 1, 32) >> bit) & 1))
            s = i32(b[:, 96:108])
            lo = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
            hi = torch.cat([(s[:, 8:12] >> (2 * j)) & 3 for j in range(4)], 1)
            sc = ((lo | (hi << 4)) - 32).double().view(nb, 2, 4, 2, 1)
            w = f16(108).view(nb, 1, 1, 1, 1) * sc * v.view(nb, 2, 4, 2, 16)
    return w.reshape(rows, _pad256(cols))


def _books(case):
    return any(t.startswith("IQ") for t in case.get("types", K6).split(","))


def _mixed64(types, qbytes, probs, rows, cols):
    w = torch.zeros(rows, cols, dtype=torch.float64, device=DEV)
    for k, (t, q) in enumerate(zip(types, qbytes)):
        w += probs[k] * _decode64(t, q, rows, cols)[:, :cols]
    return w


def _gate_grad64(types, qbytes, probs, dw):
    """Gradient of the gate logits from dL/dW [rows, cols]."""
    dp = torch.stack([(dw * _decode64(t, q, *dw.shape)[:, :dw.shape[1]]).sum() for t, q in zip(types, qbytes)])
    return probs * (dp - (probs * dp).sum())


def exact(case, seed):
    kind = case["kind"]
    # no reference for a whole step (a 64-bit run of 24 layers and two 151936-wide heads takes far over 20 s)
    # nor for the code-book formats, whose tables only this repository holds here
    if kind == "step" or _books(case):
        return None
    s = _inputs(case, seed)
    types = case.get("types", K6).split(",")
    if kind == "dequant":
        return [_decode64(t, q, case["rows"], case["cols"]) for t, q in zip(types, s["qbytes"])]
    if kind in ("linear", "routed"):
        p = torch.softmax(s["gates"].double(), 0)
        x, n, d = s["x"].double(), case["n"], case["d"]
        w = _mixed64(types, s["qbytes"], p, n, d)
        if kind == "routed":
            y = torch.zeros(case["tokens"], n, dtype=torch.float64, device=DEV)
            for k, (t, q) in enumerate(zip(types, s["qbytes"])):
                rows = (s["routing"] == k).nonzero().view(-1)
                y[rows] = x[rows] @ _decode64(t, q, n, d)[:, :d].t()
        else:
            y = x @ w.t()
        if kind == "linear" and not case["grad"]:
            return {"y": y}
        dy = s["dy"].double()
        return {"y": y, "dx": dy @ w, "dgates": _gate_grad64(types, s["qbytes"], p, dy.t() @ x)}
    if kind == "mlp":
        x, dy, m = s["x"].double(), s["dy"].double(), case["mlp"]
        shape = {"gate": (m, case["hidden"]), "up": (m, case["hidden"]), "down": (case["hidden"], m)}
        p = {k: torch.softmax(g.double(), 0) for k, (_, g) in s["tensors"].items()}
        w = {k: _mixed64(types, q, p[k], *shape[k]) for k, (q, _) in s["tensors"].items()}
        r = torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)
        norm = x * r
        g, u = norm @ w["gate"].t(), norm @ w["up"].t()
        sg = torch.sigmoid(g)
        h = g * sg * u
        dh = dy @ w["down"]
        dg, du = dh * u * sg * (1 + g * (1 - sg)), dh * g * sg
        dn = dg @ w["gate"] + du @ w["up"]
        dx = dy + r * (dn - norm * (dn * norm).mean(-1, keepdim=True))
        dw = {"gate": dg.t() @ norm, "up": du.t() @ norm, "down": dy.t() @ h}
        return {"y": x + h @ w["down"].t(), "dx": dx,
                "dgates": [_gate_grad64(types, s["tensors"][k][0], p[k], dw[k]) for k in ("gate", "up", "down")]}
    if kind == "embedding":
        p = torch.softmax(s["gates"].double(), 0)
        dim, dy = case["dim"], s["dy"].double()
        rows = [_decode64(t, q.view(case["vocab"], -1)[s["ids"]].reshape(-1), case["ids"], dim)[:, :dim]
                for t, q in zip(types, s["qbytes"])]
        y = sum(p[k] * r for k, r in enumerate(rows))
        dp = torch.stack([(dy * r).sum() for r in rows])
        return {"y": y, "dgates": p * (dp - (p * dp).sum())}
    if kind == "attention":
        b, sl, hq, hk = case["batch"], case["seq"], case["heads"], case["kv_heads"]
        cos, sin = s["cos"].double(), s["sin"].double()
        qkv = s["qkv"].double().view(b, sl, hq + 2 * hk, 64)

        def rot(t, sign):  # [.., S, 64]
            half = torch.cat([-t[..., 32:], t[..., :32]], -1)
            return t * cos + sign * half * sin

        out = torch.empty(b, hq, sl, 64, dtype=torch.float64, device=DEV)
        dqkv = torch.zeros(b, sl, hq + 2 * hk, 64, dtype=torch.float64, device=DEV)
        hide = torch.ones(sl, sl, dtype=torch.bool, device=DEV).triu(1)
        for i in range(b):
            for h in range(hq):
                j = h // (hq // hk)
                q, k, v = rot(qkv[i, :, h], 1), rot(qkv[i, :, hq + j], 1), qkv[i, :, hq + hk + j]
                pr = torch.softmax((q @ k.t() / 8.0).masked_fill(hide, -math.inf), -1)
                o, do = pr @ v, s["dout"][i, :, h].double()
                out[i, h] = o
                ds = pr * (do @ v.t() - (do * o).sum(-1, keepdim=True)) / 8.0
                dqkv[i, :, h] = rot(ds @ k, -1)
                dqkv[i, :, hq + j] += rot(ds.t() @ q, -1)
                dqkv[i, :, hq + hk + j] += pr.t() @ do
        return {"out": out, "dqkv": dqkv.view(b * sl, -1)}
    # loss
    t, v = case["temperature"], case["vocab"]
    live = int((s["labels"] >= 0).sum())
    ce = kl = 0.0
    grad = torch.empty(case["rows"], v, dtype=torch.float64, device=DEV)
    for r0 in range(0, case["rows"], 256):
        z, zt = s["logits"][r0:r0 + 256].double(), s["teacher"][r0:r0 + 256].double()
        lab = s["labels"][r0:r0 + 256]
        ls, lst, ltt = z.log_softmax(-1), (z / t).log_softmax(-1), (zt / t).log_softmax(-1)
        keep = (lab >= 0).double().view(-1, 1)
        hot = torch.zeros_like(z).scatter_(1, lab.clamp_min(0).view(-1, 1), keep)
        ce = ce - (ls * hot).sum() / live
        kl = kl + (ltt.exp() * (ltt - lst)).sum() * t * t / case["rows"]
        grad[r0:r0 + 256] = (ls.exp() * keep - hot) / live + (lst.exp() - ltt.exp()) * t / case["rows"]
    return {"ce": ce, "kl": kl, "dlogits": grad}
