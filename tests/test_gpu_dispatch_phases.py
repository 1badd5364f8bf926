"""Later phases of a dispatch called by themselves, on whatever path the sizes give the whole call: one launch (a token a
block, several, a wave by itself), separate launches with the scales in place or transposed.  After an all-phases call, after
one of the same tensors with other contents, after another shape; poisoned outputs come back bit for bit as the oracle's."""
import pytest
import torch

from mooncake_amd import _lib, ep
from mooncake_amd.harness import WorldHarness
from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, compare_dispatch

pytestmark = pytest.mark.gpu

CASES = [
    EPConfig("wave_alone", 1, 40, 640, 8, 4, True),
    EPConfig("token_a_block", 4, 64, 1024, 16, 8, True),
    EPConfig("tokens_a_block", 1, 640, 2048, 16, 8, True),
    EPConfig("tokens_a_block_bf16", 2, 300, 1024, 16, 8, False),
    EPConfig("scales_in_place", 1, 1024, 4224, 8, 5, True),
    EPConfig("separate", 2, 1032, 3072, 8, 8, True),
]


def poison(h):
    h.recv_x.fill_(0xA5 if h.cfg.use_fp8 else 0xA5A5 - 65536)
    h.src_info.fill_(-7)
    if h.cfg.use_fp8:
        h.recv_scales_phys.fill_(float("nan"))


@pytest.mark.parametrize("cfg", CASES, ids=[c.name for c in CASES])
def test_later_phases_by_themselves(gpu_device, oracle, cfg):
    world = ep.World(cfg.num_ranks)
    # more rows per expert, in more tokens of less hidden, by the separate launches: what the scratch must not be read as
    larger = EPConfig("larger", cfg.num_ranks, 2048, 640, cfg.num_experts, 4, True)
    other = WorldHarness(larger, world=world)
    other.load(generate(larger, seed=90))
    other.alloc_dispatch_outputs()
    h = WorldHarness(cfg, world=world)
    h.load(generate(cfg, seed=91))
    h.alloc_dispatch_outputs(poison=True)
    h.alloc_combine_io()
    for seed in (92, 93):
        announce(f"later phases by themselves {cfg} seed={seed}")
        data = generate(cfg, seed=seed)
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
        other.dispatch()
        h.dispatch()                                     # the last iteration's contents
        h.x.copy_(data["x"])
        h.topk_idx.copy_(data["topk_idx"])
        h.topk_weights.copy_(data["topk_weights"])
        for phases in (_lib.PHASE_FINISH, _lib.PHASE_DATA | _lib.PHASE_FINISH, _lib.PHASE_DATA):
            poison(h)
            h.dispatch()
            if cfg.use_fp8:
                h.recv_scales_phys.fill_(float("nan"))
            if phases & _lib.PHASE_DATA:
                poison(h)
            h.dispatch(phases=phases)
            if phases == _lib.PHASE_DATA and cfg.use_fp8:
                h.dispatch(phases=_lib.PHASE_FINISH)
            torch.cuda.synchronize()
            compare_dispatch(h, ref, check_poison=True)
            h.cast_back()
            h.combine()                                  # (rows by what the phases left)
            torch.cuda.synchronize()
            want = oracle.combine(h.expert_out.cpu(), data["topk_idx"], data["topk_weights"], ref["src_info"],
                                  ref["layout_range"], h.num_tokens, cfg.max_tokens, cfg.num_experts)
            assert torch.equal(h.combined.cpu().view(torch.int16), want.view(torch.int16)), (seed, phases)


def test_recorded_later_phase_goes_on_from_eager_dispatches(gpu_device, oracle):
    """A graph that holds the last phase alone: the eager calls in front of its replays leave it what it reads."""
    cfg = EPConfig("recorded_finish", 1, 640, 1024, 16, 8, True)
    announce(f"recorded last phase {cfg}")
    h = WorldHarness(cfg, world=ep.World(1))
    h.load(generate(cfg, seed=94))
    h.alloc_dispatch_outputs(poison=True)
    h.dispatch(phases=_lib.PHASE_LAYOUT | _lib.PHASE_DATA)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        h.dispatch(phases=_lib.PHASE_FINISH)
    for seed in (95, 96, 97):
        data = generate(cfg, seed=seed)
        h.x.copy_(data["x"])
        h.topk_idx.copy_(data["topk_idx"])
        poison(h)
        h.dispatch()
        h.recv_scales_phys.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, True)
        compare_dispatch(h, ref, check_poison=True)


def test_last_phase_after_replays_of_another_call(gpu_device, oracle):
    """Replays of a recorded call, which are not seen from the host, fill the world's scratch between a complete call and a
    later phase of it by itself."""
    world = ep.World(1)
    cfg = EPConfig("eager", 1, 1024, 4224, 8, 5, True)
    announce(f"last phase after replays {cfg}")
    other = WorldHarness(EPConfig("recorded", 1, 1024, 4224, 8, 5, True), world=world)     # (the same shape, other tensors)
    other.load(generate(cfg, seed=98))
    other.alloc_dispatch_outputs()
    other.dispatch()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        other.dispatch()
    h = WorldHarness(cfg, world=world)
    h.alloc_dispatch_outputs(poison=True)
    for seed in (99, 100, 101):
        data = generate(cfg, seed=seed)
        h.load(data)
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, True)
        poison(h)
        h.dispatch()
        g.replay()
        h.recv_scales_phys.fill_(float("nan"))
        h.dispatch(phases=_lib.PHASE_FINISH)
        torch.cuda.synchronize()
        compare_dispatch(h, ref, check_poison=True)
