"""Where a call's rank table comes from: kernel arguments (up to 288 words: 36 ranks of a dispatch, 32 of a combine),
memory for larger worlds, or nowhere when every tensor is evenly spaced.  Two sets of tensors take turns on one world,
so that every call finds another call's table behind it, on both sides of each limit, against the oracle."""
import pytest
import torch

from mooncake_amd import _lib, ep
from mooncake_amd.harness import WorldHarness
from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, compare_dispatch

pytestmark = pytest.mark.gpu


def _harness(cfg, world, seed, num_tokens):
    h = WorldHarness(cfg, world=world, num_tokens=num_tokens)
    h.data = generate(cfg, seed=seed)
    h.load(h.data)
    h.alloc_dispatch_outputs(poison=True)
    h.alloc_combine_io()
    h.expert_out.normal_(generator=torch.Generator(device="cuda").manual_seed(seed))
    return h


def _check(h, oracle, combined):
    cfg = h.cfg
    ref = oracle.dispatch(h.data["x"], h.data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
    compare_dispatch(h, ref, check_poison=True)
    want = oracle.combine(h.expert_out.cpu(), h.data["topk_idx"], h.data["topk_weights"], ref["src_info"],
                          ref["layout_range"], h.num_tokens, cfg.max_tokens, cfg.num_experts)
    for r, n in enumerate(h.num_tokens):
        assert torch.equal(combined[r, :n].view(torch.int16), want[r, :n].view(torch.int16)), f"rank {r}"


@pytest.mark.parametrize("uniform", [1, 0])
@pytest.mark.parametrize("ragged", [False, True], ids=["full", "ragged"])
@pytest.mark.parametrize("ranks", [1, 8, 9, 32, 33, 36, 37])
def test_calls_take_turns_on_one_world(gpu_device, oracle, ranks, ragged, uniform):
    cfg = EPConfig("tables", ranks, 8, 256, 2 * ranks, 2, True)
    nt = [(r * 5) % 9 for r in range(ranks)] if ragged else None
    announce(f"rank tables ranks={ranks} ragged={ragged} uniform={uniform}")
    world = ep.World(ranks)
    world.set_option("uniform", uniform)
    world.set_option("fused_small", 0)
    a, b = _harness(cfg, world, 1, nt), _harness(cfg, world, 2, nt)
    for _ in range(2):
        a.dispatch()
        b.dispatch(phases=_lib.PHASE_LAYOUT)
        b.dispatch(phases=_lib.PHASE_DATA)
        b.dispatch(phases=_lib.PHASE_FINISH)
        b.combine()                       # the last dispatch's handle
        a.combine()                       # an older one
        torch.cuda.synchronize()
        for h in (a, b):
            _check(h, oracle, h.combined.cpu())
        plain = b.combined.clone()
        b.expert_out.zero_()              # the packed combine must not look here
        b.cast_back()
        b.combine()
        want = b.combined.clone()
        b.combine_packed()
        torch.cuda.synchronize()
        for r, n in enumerate(b.num_tokens):
            assert torch.equal(b.combined[r, :n].view(torch.int16), want[r, :n].view(torch.int16))
        b.expert_out.normal_(generator=torch.Generator(device="cuda").manual_seed(2))
        b.combined.copy_(plain)


@pytest.mark.parametrize("search", [256, 0], ids=["searched", "resolved"])
@pytest.mark.parametrize("ranks", [3, 33])
def test_a_table_left_in_memory_is_the_next_call_s(gpu_device, oracle, ranks, search):
    """The same combine again finds its table in memory; a recorded one neither uses nor disturbs it."""
    cfg = EPConfig("left", ranks, 8, 256, 2 * ranks, 2, True)
    nt = [(r * 5) % 8 + 1 for r in range(ranks)]                # (uneven counts: the kernels read the table)
    announce(f"rank table left in memory ranks={ranks} search={search}")
    world = ep.World(ranks)
    world.set_option("combine_search_tokens", search)
    a, b = _harness(cfg, world, 3, nt), _harness(cfg, world, 4, nt)
    factor = torch.rand(cfg.num_experts, device="cuda") + 0.5
    for h in (a, b):
        h.dispatch()
        h.combine()
        h.combine_packed(factor)
    a.dispatch()
    a.combine()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    recorded = torch.empty_like(b.combined)
    with torch.cuda.graph(graph):
        b.combine()
        recorded.copy_(b.combined)
    for turn in range(3):
        for h in (a, a, b, b, a):
            h.combined.fill_(7.0)
            h.combine()
            torch.cuda.synchronize()
            _check(h, oracle, h.combined.cpu())
            if turn:
                recorded.fill_(7.0)
                graph.replay()
                torch.cuda.synchronize()
                _check(b, oracle, recorded.cpu())
            rows = h.expert_out.clone()
            h.cast_back(factor)
            h.combine()
            want = h.combined.clone()
            h.combine_packed(factor)
            torch.cuda.synchronize()
            assert torch.equal(h.combined.view(torch.int16), want.view(torch.int16))
            h.expert_out.copy_(rows)


@pytest.mark.parametrize("source", ["dispatch", "searched", "resolved"])
@pytest.mark.parametrize("ranks", [3, 32])
def test_a_table_is_left_by_a_block_without_tokens(gpu_device, oracle, ranks, source):
    """The waves of the first block end early where the first rank has no tokens; the table is in memory all the same."""
    cfg = EPConfig("left_early", ranks, 8, 256, 2 * ranks, 2, True)
    nt = [0] + [(r * 5) % 8 + 1 for r in range(1, ranks)]
    announce(f"rank table left by an empty block ranks={ranks} {source}")
    world = ep.World(ranks)
    world.set_option("combine_search_tokens", 0 if source == "resolved" else 256)
    a, b = _harness(cfg, world, 5, nt), _harness(cfg, world, 6, nt)
    a.dispatch()
    b.dispatch()
    if source == "dispatch":
        a.dispatch()
    for h in (a, a, b, b, a, a):
        h.combined.fill_(7.0)
        h.combine()
        torch.cuda.synchronize()
        _check(h, oracle, h.combined.cpu())
    rows = a.expert_out.clone()
    a.cast_back()
    a.combine()
    want = a.combined.clone()
    a.expert_out.copy_(rows)
    for _ in range(2):
        a.combined.fill_(7.0)
        a.combine_packed()
        torch.cuda.synchronize()
        for r, n in enumerate(a.num_tokens):
            assert torch.equal(a.combined[r, :n].view(torch.int16), want[r, :n].view(torch.int16))
