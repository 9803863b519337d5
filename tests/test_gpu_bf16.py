"""The kernel's bf16 rounding, bit for bit: round to nearest even over every
bf16 weight, and one NaN pattern (0x7fc0) in every tensor a launch writes,
whatever sign and payload the NaN it came from had."""

import pytest
import torch

from full_harness import FullCase
from llama_harness import LlamaCase
from megakernels_amd.latency.synthetic import LlamaConfig
from megakernels_amd.mixtral.synthetic import TINY, MoEConfig, with_layers
from moe_harness import MoECase

pytestmark = pytest.mark.gpu
NAN = 0x7FC0
ODD_NAN = 0xFFE5 - 0x10000  # negative, quiet, with a payload (as int16)


def bits(t):
    return t.detach().contiguous().view(torch.int16).cpu().to(torch.int32) & 0xFFFF


def round_bf16(f):
    """bf16 bits of an fp32 tensor, by integers."""
    u = f.contiguous().view(torch.int32).to(torch.int64) & 0xFFFFFFFF
    r = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16) & 0xFFFF
    return torch.where(torch.isnan(f), torch.full_like(r, NAN), r).to(torch.int32)


def unit_rms_residual(H, gen):
    """H multiples of 1/16 below 2 whose squares add up to exactly H (every
    partial sum of them is exact in fp32), so that the norm's factor is 1."""
    k = torch.randint(8, 24, (H - 4,), generator=gen)
    target = 256 * H
    i = 0
    while int((k * k).sum()) > target:
        k[i], i = 8, i + 1
    while target - int((k * k).sum()) > 961:
        i = int(torch.randint(0, H - 4, (1,), generator=gen))
        k[i] += 1 if k[i] < 24 and target - int((k * k).sum()) >= 2 * int(k[i]) + 1 else 0
    rest = target - int((k * k).sum())
    tail = next((a, b, c, d) for a in range(32) for b in range(32) for c in range(32) for d in range(32)
                if a * a + b * b + c * c + d * d == rest)
    return (torch.cat([k, torch.tensor(tail)])[torch.randperm(H, generator=gen)] / 16).to(torch.bfloat16)


def test_norm_rounds_every_weight():
    """normed = bf16(w * bf16(x * r)) with r = 1: products of every bf16
    pattern (denormals, infinities and NaNs among them) and multiples of 1/16,
    ties included."""
    H = 4096
    case = MoECase(MoEConfig(1, H, 512, 8, 2, 2, 2, 64, rms_norm_eps=0.0), seed=1)
    gen = torch.Generator().manual_seed(2)
    patterns = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    for part in patterns.split(H):
        x = unit_rms_residual(H, gen)
        w = part[torch.randperm(H, generator=gen)]
        case.g_gpu.ffn_ln_weights[0].copy_(w)
        case.reset(x)
        case.run_gpu()
        want = round_bf16(w.float() * x.float())
        got = bits(case.g_gpu.router_normed_hidden)
        assert torch.equal(got, want), [(hex(int(a)), hex(int(b))) for a, b in zip(got, want) if a != b][:4]


def _one_pattern(tensors, nan):
    """The tensors named in `nan` hold NaNs, and every NaN is 0x7fc0."""
    for name, t in tensors.items():
        here = torch.isnan(t).cpu()
        assert bool(here.any()) or name not in nan, f"{name}: no NaN"
        odd = bits(t)[here] != NAN
        assert not bool(odd.any()), f"{name}: {[hex(int(v)) for v in bits(t)[here][odd][:4]]}"


@pytest.mark.parametrize("where,nan", [("residual", ("normed", "scores", "silu", "hidden")),
                                       ("norm", ("normed", "scores", "silu", "hidden")),
                                       ("gate", ("silu", "hidden")), ("down", ("hidden",))])
def test_moe_stores_one_nan(where, nan):
    case = MoECase(MoEConfig(1, 512, 512, 8, 2, 3, 2, 64), seed=5)
    g = case.g_gpu
    x = torch.randn(512, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16)
    if where == "residual":
        x.view(torch.int16)[77] = ODD_NAN
    elif where == "norm":
        g.ffn_ln_weights.view(torch.int16)[0, 40] = ODD_NAN
    elif where == "gate":
        g.expert_gate_weights.view(torch.int16)[0, :, 9, 3] = ODD_NAN
    else:
        g.expert_down_weights.view(torch.int16)[0, :, 9, 3] = ODD_NAN
    case.reset(x)
    case.run_gpu()
    _one_pattern({"normed": g.router_normed_hidden, "scores": g.selected_expert_scores, "silu": g.expert_silu_out,
                  "hidden": g.hidden_states}, nan)


@pytest.mark.parametrize("where,nan", [("q", ("q",)), ("k", ("k",)),
                                       ("v", ("v", "attn_out", "hidden", "silu", "logits")),
                                       ("o", ("hidden", "silu", "logits")), ("down", ("hidden", "logits")),
                                       ("lm_head", ("logits",))])
@pytest.mark.parametrize("cached,hidden", [(5, 512), (300, 1024)])
def test_dense_stores_one_nan(where, nan, cached, hidden):
    """One partition and several; the LM head's fallback and its row items."""
    case = LlamaCase(LlamaConfig(1, hidden, 512, hidden // 64, hidden // 64, 64), seed=7, prefill=cached, steps=1)
    g = case.g_gpu
    row = {"q": 9, "k": hidden + 9, "v": 2 * hidden + 9}.get(where, 9)
    w = {"o": g.o_proj_weights[0], "down": g.down_proj_weights[0], "lm_head": g.lm_head_weights}.get(
        where, g.qkv_proj_weights[0])
    w.view(torch.int16)[row, 3] = ODD_NAN
    case.step(3)
    _one_pattern({"q": g.post_ln_rope_q, "k": g.k_cache, "v": g.v_cache, "attn_out": g.attn_out,
                  "hidden": g.hidden_states, "silu": g.silu_out, "logits": g.logits}, nan)


def test_mixtral_logits_store_one_nan():
    """The Mixtral LM head adds its column blocks with packed atomics."""
    case = FullCase(with_layers(TINY, 1), seed=8, prefill=5, steps=1)
    case.g_gpu.lm_head_weights.view(torch.int16)[9, 3] = ODD_NAN
    case.step(3)
    _one_pattern({"logits": case.g_gpu.logits, "hidden": case.g_gpu.hidden_states}, ("logits",))
