"""GPU parity: the persistent HIP kernel against the CPU oracle.

Every test launches through the reference-shaped ``mk_mixtral`` launcher
(ctypes -> C ABI ``mk_mixtral_launch``), with ``debug_sync=True`` so a
device-side failure raises.  Bar: expert indices exact, hidden / SiLU /
normed within max-abs-rel 2e-2, normed and SiLU within one bf16 ulp, at
least 99 % of hidden / SiLU / normed bit-identical (``moe_harness``), barrier
tensor equal to the oracle's.
"""

import pytest
import torch

from megakernels_amd.mixtral.synthetic import C1, C2, SMALL
from moe_harness import MoECase, assert_bf16_close, draw_tokens

pytestmark = pytest.mark.gpu


def _report(name, res):
    print(f"[{name}] experts {res.indices_gpu} hidden {res.err_hidden:.2e} silu {res.err_silu:.2e} "
          f"normed {res.err_normed:.2e}", flush=True)


@pytest.fixture(scope="module")
def c1_case():
    return MoECase(C1, seed=0)


def test_library_loads_on_gpu():
    import mk_mixtral

    cus, max_workers = mk_mixtral.query_device("cuda:0")
    assert cus == torch.cuda.get_device_properties(0).multi_processor_count
    assert max_workers >= cus


def test_c1_first_token(c1_case):
    tokens = draw_tokens(c1_case.cpu_model, 1)
    res = c1_case.run_token(tokens[0])
    _report("c1 token 0", res)
    res.assert_ok()


def test_c1_64_tokens(c1_case):
    """Config 1: 64 independent decode tokens, seed 0, margin rule."""
    tokens = draw_tokens(c1_case.cpu_model, 64)
    worst = 0.0
    for t in range(tokens.shape[0]):
        res = c1_case.run_token(tokens[t])
        res.assert_ok()
        worst = max(worst, res.err_hidden, res.err_silu)
    print(f"[c1 x64] worst max-abs-rel {worst:.2e}", flush=True)


def test_reference_small_shapes_random_norm_weights():
    """The reference debug shapes (H 512, F 1024, E 4) with non-unit RMSNorm
    weights, which exercise the second bf16 rounding of the norm."""
    case = MoECase(SMALL, seed=42, ln_weight_std=0.1)
    for x in draw_tokens(case.cpu_model, 8):
        res = case.run_token(x)
        _report("small", res)
        res.assert_ok()


@pytest.mark.parametrize("ebs,dbs", [(16, 16), (8, 4), (4, 8)])
def test_block_sizes(ebs, dbs):
    """(16, 16) is the reference's own partition."""
    case = MoECase(C1, seed=3, expert_proj_block_size=ebs, down_proj_block_size=dbs)
    for x in draw_tokens(case.cpu_model, 2):
        case.run_token(x).assert_ok()


@pytest.mark.parametrize("mode", ["zz", "wave", "dag"])
def test_assignment_modes(mode):
    case = MoECase(C1, seed=5, mode=mode)
    for x in draw_tokens(case.cpu_model, 2):
        case.run_token(x).assert_ok()


@pytest.mark.parametrize("workers", [1, 7, 64])
def test_fewer_workers(workers):
    """Fewer workers than compute units: longer queues per worker."""
    case = MoECase(SMALL, seed=9, workers=workers)
    x = draw_tokens(case.cpu_model, 1)[0]
    case.run_token(x).assert_ok()


def test_upgate_only_stage():
    """stop_after_op='rms_router_upgate' (the reference's stage test)."""
    case = MoECase(C1, seed=11, stop_after_op="rms_router_upgate")
    x = draw_tokens(case.cpu_model, 1)[0]
    res = case.run_token(x)
    res.assert_ok()


def test_skewed_router_bias():
    """+2.0 router bias on experts 0 and 1 (config 2's skewed variant, at
    config 1 shapes)."""
    bias = [2.0, 2.0] + [0.0] * (C1.num_local_experts - 2)
    case = MoECase(C1, seed=0, router_bias=bias)
    hits = 0
    for x in draw_tokens(case.cpu_model, 8):
        res = case.run_token(x)
        res.assert_ok()
        hits += sum(i in (0, 1) for i in res.indices_ref)
    assert hits >= 12  # the bias makes experts 0 and 1 dominate


def test_speculative_predict():
    """Opcode 8 with a noisy predictor copy of the router."""
    case = MoECase(C1, seed=0, predict=True, predictor_sigma=0.01)
    for x in draw_tokens(case.cpu_model, 4):
        res = case.run_token(x)
        res.assert_ok()
        assert res.predicted_gpu == res.predicted_ref


def test_deterministic_relaunch(c1_case):
    x = draw_tokens(c1_case.cpu_model, 1)[0]
    c1_case.reset(x)
    c1_case.run_gpu()
    first = c1_case.g_gpu.hidden_states.clone()
    c1_case.reset(x)
    c1_case.run_gpu()
    assert torch.equal(first, c1_case.g_gpu.hidden_states)


def test_timings_recorded(c1_case):
    x = draw_tokens(c1_case.cpu_model, 1)[0]
    c1_case.reset(x)
    c1_case.g_gpu.timings.zero_()
    c1_case.run_gpu(record_timings=True)
    t = c1_case.g_gpu.timings.cpu().to(torch.int64) & 0xFFFFFFFF
    ops = c1_case.g_gpu.instructions[:, :, 0].cpu()
    busy = ops != 0
    assert bool((t[:, :, 0][busy] > 0).all())
    assert bool((t[:, :, 4][busy] >= t[:, :, 0][busy]).all())


@pytest.mark.slow
def test_c2_tokens():
    """Config 2 shapes (H 4096, F 14336, E 8): a few tokens."""
    case = MoECase(C2, seed=0, generate_on_device=True)
    for x in draw_tokens(case.cpu_model, 3):
        res = case.run_token(x)
        _report("c2", res)
        res.assert_ok()


@pytest.mark.parametrize("config,workers,mode", [("c1", None, "rr"), ("small", None, "rr"), ("small", 7, "rr"),
                                                 ("small", 1, "rr"), ("c1", None, "dag"), ("c1", 20, "zz")])
def test_work_sharing(config, workers, mode):
    """Pooled opcode-5 items (groups of consecutive workers share one claim
    counter): same results and barrier counts as the static partition."""
    cfg = C1 if config == "c1" else SMALL
    case = MoECase(cfg, seed=13, workers=workers, mode=mode, predict=(mode == "dag"))
    for x in draw_tokens(case.cpu_model, 3):
        res = case.run_token(x, work_sharing=True)
        res.assert_ok()


def test_work_sharing_more_instructions_than_the_pool():
    """Work sharing on a schedule whose groups hold more opcode-5
    instructions than one pool lists (one instruction per block,
    interleaved: about 45 per worker, ~358 per group of 8 workers at 20
    workers, of which a pool lists the at most 64 near one queue depth):
    owners finish alone what no one near them lists, and every instruction
    arrives once."""
    case = MoECase(C1, seed=19, workers=20, mode="zz", moe_overlap=True, ln_weight_std=0.1)
    per_worker = (case.g_gpu.instructions[:, :, 0] == 5).sum(dim=1)
    assert int(per_worker[:8].sum()) > 64
    for x in draw_tokens(case.cpu_model, 3):
        res = case.run_token(x, work_sharing=True)
        _report("work-sharing pool overflow", res)
        res.assert_ok()


@pytest.mark.parametrize("config", ["c1", "small"])
def test_speed_balanced_partition(config):
    """Row partitions re-split by per-worker speed (odd XCDs slower), block
    size 1: same results and barrier totals as the oracle's even partition."""
    cfg = C1 if config == "c1" else SMALL
    W = torch.cuda.get_device_properties(0).multi_processor_count
    weights = [1.07 if w % 2 == 0 else 0.93 for w in range(W)]
    case = MoECase(cfg, seed=17, expert_proj_block_size=1, down_proj_block_size=1, worker_weights=weights)
    for x in draw_tokens(case.cpu_model, 3):
        case.run_token(x).assert_ok()
        case.run_token(x, work_sharing=True).assert_ok()


@pytest.mark.parametrize("config,workers,mode,ebs", [("c1", None, "rr", None), ("c1", None, "rr", 4),
                                                     ("c1", 64, "rr", None), ("c1", 1, "rr", None),
                                                     ("c1", 20, "zz", None), ("c1", None, "dag", None),
                                                     ("small", 7, "rr", None)])
def test_moe_overlap(config, workers, mode, ebs):
    """Interleaved opcode-5 partition (pooled instructions, per-item arrivals)
    with opcode 6 starting on finished column groups: indices exact, hidden
    and SiLU within tolerance, barrier tensor equal to the oracle's, over
    consecutive launches (the chunk counters are cleared at each launch's
    end).  C1 (F = 3584: 7 chunks) ends in a short group of 3; SMALL has 4
    experts, so only the pooled opcode 5 applies there."""
    cfg = C1 if config == "c1" else SMALL
    case = MoECase(cfg, seed=21, workers=workers, mode=mode, predict=(mode == "dag"), moe_overlap=True,
                   expert_proj_block_size=ebs)
    for x in draw_tokens(case.cpu_model, 3):
        res = case.run_token(x)
        _report(f"overlap-{config}-{workers}-{mode}-{ebs}", res)
        res.assert_ok()
        # opcode 6 adds its column groups in a fixed order whatever the
        # order they became ready in: a relaunch is bit-identical, and the
        # launch without the overlap differs in fp32 summation order only
        first = case.g_gpu.hidden_states.clone()
        case.reset(x)
        case.run_gpu()
        assert torch.equal(case.g_gpu.hidden_states, first), "overlapped relaunch is not bit-identical"
        case.reset(x)
        case.run_gpu(downproj_overlap=False)
        assert_bf16_close("hidden, overlap on vs off", first, case.g_gpu.hidden_states, max_ulp=2)


def test_moe_overlap_mixed_launches():
    """Overlap on the reference's contiguous partition, then off, then with
    work sharing (which turns it off), then on again: every launch matches
    the oracle, so no launch leaves counters behind for the next."""
    case = MoECase(C1, seed=23)
    xs = draw_tokens(case.cpu_model, 4)
    for x, kw in zip(xs, ({"downproj_overlap": True}, {}, {"downproj_overlap": True, "work_sharing": True},
                          {"downproj_overlap": True})):
        case.run_token(x, **kw).assert_ok()


def test_moe_overlap_c2_tokens():
    """Config 2 shapes with the overlap: a few tokens."""
    case = MoECase(C2, seed=0, generate_on_device=True, moe_overlap=True)
    for x in draw_tokens(case.cpu_model, 3):
        res = case.run_token(x)
        _report("c2-overlap", res)
        res.assert_ok()
