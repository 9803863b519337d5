"""Performance cases of the decode megakernels.

Every case is one call (or a few) of a public entry point as a decoding
program makes it: one MoE layer, one attention block, one decoder layer
(``interpret`` over a schedule of ``make_moe_dag`` / ``make_dag``), or decode
steps of a model (``MK_Generator.run``).  Decoding is batch 1, so a pass reads
every weight it uses once; a program's inputs are the residual stream or the
token ids it writes before the call.

Weights are random bf16 of the named shapes (the package's own synthetic
models), the KV cache is filled with N(0, 1) up to ``cached`` positions.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "epic-kernel_amd"))

from megakernels_amd.latency import mk as llama_mk  # noqa: E402
from megakernels_amd.latency import scheduler as llama_sched  # noqa: E402
from megakernels_amd.latency.synthetic import LlamaConfig, make_synthetic_llama  # noqa: E402
from megakernels_amd.mixtral import mk as moe_mk  # noqa: E402
from megakernels_amd.mixtral import scheduler as moe_sched  # noqa: E402
from megakernels_amd.mixtral.generate import MK_Generator  # noqa: E402
from megakernels_amd.mixtral.synthetic import MoEConfig, make_synthetic_mixtral  # noqa: E402
from megakernels_amd.scheduler import Schedule, assign_to_sms, tensorize_instructions  # noqa: E402

# kinds of case:
#   moe        one MoE layer (opcodes 5 and 6), the residual written by the caller
#   attention  QKV to the O projection of one layer
#   layer      a whole decoder layer, no LM head
#   decode     `tokens` decode steps of a whole model with its LM head


def _case(name, kind, vm, hidden, ffn, heads=8, kv_heads=2, experts=8, layers=1, vocab=512, cached=0, tokens=1):
    return {"name": name, "kind": kind, "vm": vm, "hidden": hidden, "ffn": ffn, "heads": heads, "kv_heads": kv_heads,
            "experts": experts if vm == "mixtral" else 1, "layers": layers, "vocab": vocab, "cached": cached,
            "tokens": tokens}


def listed():
    return [
        # the smallest MoE layer in use (debugging shape): all latency
        _case("moe-small", "moe", "mixtral", 512, 1024, 8, 2, experts=4),
        # a small MoE layer whose active weights fit in the caches
        _case("moe-1k", "moe", "mixtral", 1024, 3584, 8, 2),
        # many experts, sizes that are odd multiples of a 512-column chunk
        _case("moe-16-experts", "moe", "mixtral", 2560, 6656, 20, 5, experts=16),
        # one full-size Mixtral-8x7B MoE layer
        _case("moe-8x7b", "moe", "mixtral", 4096, 14336, 32, 8),
        # a short prompt in a small model: one partition, head dim 64
        _case("attention-short", "attention", "llama", 1024, 1536, 16, 4, cached=77),
        # a growing chat in the full-size model, at a position inside a block
        _case("attention-8x7b-4k", "attention", "mixtral", 4096, 14336, 32, 8, cached=4133),
        # a long document: the KV cache is most of the traffic
        _case("attention-8x7b-16k", "attention", "mixtral", 4096, 14336, 32, 8, cached=16383),
        # a small dense layer, a few hundred positions
        _case("layer-1536", "layer", "llama", 1536, 2048, 12, 4, cached=300),
        # one layer of the dense 3B model
        _case("layer-3b", "layer", "llama", 3072, 8192, 24, 8, cached=2048),
        # a two-layer model fed a short prompt token by token: launches count
        _case("decode-tiny", "decode", "llama", 1024, 1536, 16, 4, layers=2, vocab=256, cached=20, tokens=8),
        # eight layers of the dense 3B model with its LM head (bf16 roundings
        # that differ travel through every later layer: over all 28 two right
        # answers are too far apart to be compared)
        _case("decode-3b", "decode", "llama", 3072, 8192, 24, 8, layers=8, vocab=128256, cached=2048, tokens=2),
        # three layers of Mixtral-8x7B with its LM head (the whole model does
        # not fit the card three times)
        _case("decode-8x7b", "decode", "mixtral", 4096, 14336, 32, 8, layers=3, vocab=32000, cached=4096, tokens=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Sizes over the ranges above: hidden 512 to 4096 and FFN 1024 to 14336
    in 512-column chunks, 2 to 16 experts, 1 to 16383 cached positions (a
    whole model at most 4096), 1 to 4 query heads per KV head."""
    kind = rng.choice(["moe", "attention", "layer", "decode"])
    vm = "mixtral" if kind == "moe" else rng.choice(["mixtral", "llama"])
    ffn = 512 * _log_int(rng, 2, 28)
    if kind == "decode" and vm == "mixtral":
        hidden = rng.choice([2048, 4096])  # the Mixtral LM head reduces in 2048-column blocks
    else:
        hidden = 512 * rng.randint(1, 8)
    head_dim = rng.choice([64, 128])
    heads = hidden // head_dim
    kv_heads = heads // rng.choice([g for g in (1, 2, 3, 4) if heads % g == 0])
    if kind == "decode":
        layers = rng.randint(1, 3) if vm == "mixtral" else rng.randint(1, 8)
        cached, vocab, tokens = _log_int(rng, 1, 4096), 16 * _log_int(rng, 16, 2000), rng.randint(1, 2)
    else:
        layers, vocab, tokens = 1, 512, 1
        cached = 0 if kind == "moe" else _log_int(rng, 1, 16383)
    case = _case("", kind, vm, hidden, ffn, heads, kv_heads, experts=rng.choice([2, 4, 6, 8, 8, 16]), layers=layers,
                 vocab=vocab, cached=cached, tokens=tokens)
    del case["name"]
    return case


def _model(case, seed):
    full = case["kind"] != "moe"
    shape = (case["layers"], case["hidden"], case["ffn"], case["heads"], case["kv_heads"])
    kv = case["cached"] + case["tokens"]
    if case["vm"] == "llama":
        return make_synthetic_llama(LlamaConfig(*shape, case["vocab"]), "cuda", seed, ln_weight_std=0.1,
                                    kv_positions=kv, prefill=case["cached"])
    # decode steps: skewed routing (+2 on two experts) and the speculative
    # predictor's weights (router + noise), as the benchmark's configurations
    bias = [2.0, 2.0] + [0.0] * (case["experts"] - 2) if case["kind"] == "decode" else None
    return make_synthetic_mixtral(MoEConfig(*shape, case["experts"], 2, case["vocab"]), "cuda", seed,
                                  ln_weight_std=0.1, router_bias=bias,
                                  predictor_sigma=0.003 if case["kind"] == "decode" else None, full=full,
                                  kv_positions=kv, prefill=case["cached"])


def _residual(case, model, seed):
    """A residual N(0, 1).  A near tie in the router has two right answers, so
    an MoE input is the one of a few whose second and third logits are
    furthest apart."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed + 77)
    x = torch.empty([16, case["hidden"]], dtype=torch.bfloat16, device="cuda").normal_(0.0, 1.0, generator=gen)
    if case["kind"] == "attention" or case["experts"] <= 2:
        return x[0].clone()
    sp = model.stacked_params
    xf = x.float()
    n = xf * torch.rsqrt(xf.square().mean(1, keepdim=True) + 1e-5) * sp.ffn_ln_weight[0].float()
    top = (n @ sp.router_weight[0].float().t()).topk(3, dim=1).values
    return x[int((top[:, 1] - top[:, 2]).argmax())].clone()


def prepare(case, seed):
    model = _model(case, seed)
    s = SimpleNamespace(case=case, model=model)
    if case["kind"] == "decode":
        # logits of a Mixtral step stay readable only without the reset
        kw = {"reset_next": False} if case["vm"] == "mixtral" else {}
        s.gen = MK_Generator.build(model, case["cached"], **kw)
        s.g = s.gen.schedule.globs
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed + 99)
        s.ids = torch.randint(0, case["vocab"], [1, case["tokens"]], device="cuda", generator=gen)
        s.steps = [(s.ids[:, i:i + 1], case["cached"] + i) for i in range(case["tokens"])]
    else:
        mod, mk = (llama_sched, llama_mk.LatencyMK_Interpreter) if case["vm"] == "llama" else (
            moe_sched, moe_mk.MixtralMK_Interpreter)
        s.g = mod.make_globals(model, seq_len=case["cached"])
        if case["kind"] == "moe":
            nodes = mod.make_moe_dag(s.g)
        else:
            nodes = mod.make_dag(s.g, stop_after_op="oproj" if case["kind"] == "attention" else "downproj",
                                 layer_limit=1)
        tensorize_instructions(s.g, assign_to_sms("rr", schedule=Schedule(s.g, *nodes)))
        s.interpreter = mk()
        s.residual = _residual(case, model, seed) if case["vm"] == "mixtral" else torch.empty(
            case["hidden"], dtype=torch.bfloat16, device="cuda").normal_(
                0.0, 1.0, generator=torch.Generator(device="cuda").manual_seed(seed + 77))
    g = s.g
    s.out = {"hidden": g.hidden_states}
    if case["kind"] != "moe":
        lo, hi = case["cached"], case["cached"] + case["tokens"]
        s.out.update(keys=g.k_cache[:, 0, lo:hi], values=g.v_cache[:, 0, lo:hi])
    if case["kind"] == "attention":
        s.out.update(queries=g.post_ln_rope_q, attn_out=g.attn_out)
    if case["kind"] in ("moe", "layer"):
        s.out["silu"] = g.silu_out if case["vm"] == "llama" else g.expert_silu_out
    if case["kind"] in ("moe", "layer") and case["vm"] == "mixtral":
        s.out.update(normed=g.router_normed_hidden, experts=g.selected_expert_indices,
                     scores=g.selected_expert_scores)
    if case["kind"] == "decode":
        s.out["logits"] = g.logits
    return s


def run(state):
    g = state.g
    kind = state.case["kind"]
    if kind == "decode":
        # the tokens picked are not returned: of two logits that tie in bf16
        # either is a right answer; the logits they are picked from are
        for ids, pos in state.steps:
            state.gen.run(ids, pos)
        return state.out
    g.hidden_states.copy_(state.residual)
    g.barriers.zero_()
    if kind == "moe":
        moe_sched.prefill_oproj_barrier(g)
    state.interpreter.interpret(g)
    return state.out


def work(case):
    H, F, E, L, t = (case[k] for k in ("hidden", "ffn", "experts", "layers", "tokens"))
    D = H // case["heads"]
    kvd = case["kv_heads"] * D
    k = 2 if case["vm"] == "mixtral" else 1
    mlp = 3 * k * F * H + (E * H if k == 2 else 0) + H
    attn = (H + 2 * kvd) * H + H * H + H
    seq = case["cached"] + (t + 1) / 2
    weights = {"moe": mlp, "attention": attn}.get(case["kind"], L * (mlp + attn))
    kv = 0 if case["kind"] == "moe" else L * 2 * kvd * seq
    head = case["vocab"] * H + H if case["kind"] == "decode" else 0
    flops = 2 * (weights + head) + (0 if case["kind"] == "moe" else L * 4 * H * seq)
    return {"bytes": 2 * t * (weights + kv + head), "flops": t * flops}


def tolerance(case):
    # four times what one layer's bf16 roundings were seen to do (0.002 to
    # 0.007 against 64 bits; 0.016 over four whole layers and the LM head)
    return {"rel": 0.03 if case["layers"] > 1 else 0.02}


def _rms64(x, w):
    return x * torch.rsqrt(x.square().mean() + 1e-5) * w.double()


def _attention64(case, sp, layer, x, pos, keys, values, cos, sin):
    """q, attention output and the residual after the O projection; the new
    K and V rows are appended to `keys` and `values`."""
    heads, kvh = case["heads"], case["kv_heads"]
    D = case["hidden"] // heads
    qkv = sp.qkv_proj[layer].double() @ _rms64(x, sp.attn_ln_weight[layer])
    q, k, v = (t.view(-1, D) for t in qkv.split([heads * D, kvh * D, kvh * D]))
    c, s = cos[pos].double(), sin[pos].double()

    def rope(t):
        turned = torch.stack([-t[:, 1::2], t[:, 0::2]], dim=2).flatten(1)
        return t * c + turned * s

    q, k = rope(q), rope(k)
    keys.append(k)
    values.append(v)
    K = torch.cat([keys[0]] + [t[None] for t in keys[1:]]).repeat_interleave(heads // kvh, dim=1)
    V = torch.cat([values[0]] + [t[None] for t in values[1:]]).repeat_interleave(heads // kvh, dim=1)
    p = torch.softmax((K * q[None]).sum(2) / math.sqrt(D), dim=0)
    out = (p[:, :, None] * V).sum(0).flatten()
    return q.flatten(), out, x + sp.o_proj[layer].double() @ out


def _silu64(gate, up, n):
    a = gate.double() @ n
    return a * torch.sigmoid(a) * (up.double() @ n)


def _mlp64(case, sp, layer, x):
    if case["vm"] == "llama":
        h = _silu64(sp.gate_proj[layer], sp.up_proj[layer], _rms64(x, sp.mlp_ln_weight[layer]))
        return x + sp.down_proj[layer].double() @ h, {"silu": h}
    n = _rms64(x, sp.ffn_ln_weight[layer])
    logits = sp.router_weight[layer].double() @ n
    if sp.router_bias is not None:
        logits = logits + sp.router_bias[layer].double()
    top, idx = logits.topk(2)
    scores = torch.softmax(top, 0)
    silu = torch.zeros(case["experts"], case["ffn"], dtype=torch.float64, device=x.device)
    for p, e in zip(scores, idx.tolist()):
        silu[e] = _silu64(sp.expert_gate[layer, e], sp.expert_up[layer, e], n)
        x = x + p * (sp.expert_down[layer, e].double() @ silu[e])
    return x, {"silu": silu, "normed": n, "experts": idx.to(torch.int32), "scores": scores}


def exact(case, seed):
    s = prepare(case, seed)
    sp, model = s.model.stacked_params, s.model
    if case["kind"] == "moe":
        x, out = _mlp64(case, sp, 0, s.residual.double())
        return {"hidden": x, **out}
    kc, vc = model.stacked_kv_cache
    keys = [[kc[l, 0, :case["cached"]].double()] for l in range(case["layers"])]
    values = [[vc[l, 0, :case["cached"]].double()] for l in range(case["layers"])]
    rope = model.model.rope_cos, model.model.rope_sin
    out = {}
    for i in range(case["tokens"]):
        pos = case["cached"] + i
        x = (model.embed_tokens[int(s.ids[0, i])] if case["kind"] == "decode" else s.residual).double()
        for layer in range(case["layers"]):
            q, a, x = _attention64(case, sp, layer, x, pos, keys[layer], values[layer], *rope)
            if case["kind"] == "attention":
                out.update(queries=q, attn_out=a)
            else:
                x, mlp = _mlp64(case, sp, layer, x)
                if case["kind"] == "layer":
                    out.update(mlp)
    out["hidden"] = x
    out["keys"] = torch.stack([torch.stack(k[1:]) for k in keys])
    out["values"] = torch.stack([torch.stack(v[1:]) for v in values])
    if case["kind"] == "decode":
        head = model.lm_head
        out["logits"] = head.lm_head.weight.double() @ _rms64(x, head.input_norm.weight)
    return out
