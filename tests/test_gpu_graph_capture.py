"""Whole-world calls recorded into HIP graphs: every replay, on fresh input
values, must give what the oracle gives - also with eager calls of the same
world between the replays, which rewrite the world's shared tables and routing
state.  (Serving loops run dispatch / combine from graphs; the reference's
low-latency kernels are written to be capturable for that reason.)"""
import pytest
import torch

from mooncake_amd import ep
from mooncake_amd.harness import WorldHarness
from mooncake_amd.mooncake_ep_buffer import Buffer, LogicalGroup
from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, compare_dispatch

pytestmark = pytest.mark.gpu


def _reference(oracle, cfg, data, factor):
    nt = [cfg.tokens_per_rank] * cfg.num_ranks
    ref = oracle.dispatch(data["x"], data["topk_idx"], nt, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
    rows = oracle.cast_back(ref["recv_x"], ref["scales"] if cfg.use_fp8 else None, ref["recv_count"], factor)
    out = oracle.combine(rows, data["topk_idx"], data["topk_weights"], ref["src_info"], ref["layout_range"], nt,
                         cfg.max_tokens, cfg.num_experts)
    return ref, out


def _load_in_place(h, data):
    h.x.copy_(data["x"])
    h.topk_idx.copy_(data["topk_idx"])
    h.topk_weights.copy_(data["topk_weights"])


def _harness(cfg, world, seed):
    h = WorldHarness(cfg, world=world)
    h.load(generate(cfg, seed=seed))
    h.alloc_dispatch_outputs(poison=False)
    h.alloc_combine_io()
    return h


@pytest.mark.parametrize("use_fp8", [True, False])
@pytest.mark.parametrize("one_graph,search", [(True, 256), (False, 256), (False, 0)],
                         ids=["one_graph", "searched", "resolved"])
def test_replays_match_the_oracle(gpu_device, oracle, use_fp8, one_graph, search):
    cfg = EPConfig("graph", 4, 48, 1024, 16, 4, use_fp8, masked_fraction=0.2)
    announce(f"graph capture {cfg} one_graph={one_graph} search={search}")
    world = ep.World(cfg.num_ranks)
    world.set_option("combine_search_tokens", search)
    h = _harness(cfg, world, seed=100)
    other = _harness(cfg, world, seed=200)          # eager traffic on the same world
    factor = (torch.arange(cfg.num_experts, dtype=torch.float32) * 0.1 + 1.0).to(gpu_device)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):                   # sizes the world's scratch; nothing may grow while recording
        h.dispatch()
        h.cast_back(factor)
        h.combine()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()

    graphs = []
    if one_graph:                                   # combine reuses the routing state of the dispatch beside it
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            h.dispatch()
            h.cast_back(factor)
            h.combine()
        graphs = [g]
    else:                                           # a combine recorded on its own looks its handle up
        for part in (lambda: (h.dispatch(), h.cast_back(factor)), h.combine):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                part()
            graphs.append(g)
        # in the reduce kernel, or through routes: cleared, resolved, read
        assert world.get_option("last_combine_launches") == (1 if search else 3)

    for seed in (1, 2, 3):
        data = generate(cfg, seed=seed)
        _load_in_place(h, data)
        h.combined.zero_()
        other.dispatch()                            # overwrites the shared tables and the routing state
        other.cast_back(None)
        other.combine()
        torch.cuda.synchronize()
        for g in graphs:
            g.replay()
        torch.cuda.synchronize()
        ref, want = _reference(oracle, cfg, data, factor.cpu())
        compare_dispatch(h, ref, check_poison=False)
        assert torch.equal(h.combined.cpu().view(torch.int16), want.view(torch.int16)), f"replay with seed {seed}"

    # eager calls of the world are still right after its graphs ran
    data = generate(cfg, seed=200)
    ref, want = _reference(oracle, cfg, data, None)
    other.dispatch()
    other.cast_back(None)
    other.combine()
    torch.cuda.synchronize()
    compare_dispatch(other, ref, check_poison=False)
    assert torch.equal(other.combined.cpu().view(torch.int16), want.view(torch.int16))


def test_recording_refuses_to_grow_scratch_and_per_rank_calls(gpu_device):
    cfg = EPConfig("graph_refusals", 2, 16, 256, 4, 2, False)
    announce(f"graph refusals {cfg}")
    world = ep.World(cfg.num_ranks)
    h = _harness(cfg, world, seed=1)                # never called eagerly: its scratch does not exist yet
    buf = Buffer(LogicalGroup(world, 0), Buffer.get_ep_buffer_size_hint(16, 256, 2, 4))
    marker = torch.zeros(8, device=gpu_device)
    g = torch.cuda.CUDAGraph()
    errors = []
    with torch.cuda.graph(g):
        marker.add_(1.0)                            # so that the graph is not empty
        try:
            h.dispatch()
        except RuntimeError as e:
            errors.append(str(e))
        try:
            buf.dispatch(h.x[0], h.topk_idx[0], None, cfg.max_tokens, cfg.num_experts, -1, use_fp8=False)
        except NotImplementedError as e:
            errors.append(str(e))
    assert len(errors) == 2
    assert "outside the capture first" in errors[0]
    assert "cannot be recorded into a graph" in errors[1]
    g.replay()
    torch.cuda.synchronize()
    assert float(marker[0]) == 1.0
    # the refused calls left the world usable
    h.dispatch()
    torch.cuda.synchronize()
    assert int(h.recv_count.sum()) == int((h.topk_idx >= 0).sum())


@pytest.mark.parametrize("two_parts", [False, True], ids=["more_tokens", "two_parts"])
def test_a_one_launch_call_prepares_for_recording_the_others(gpu_device, oracle, two_parts):
    """An eager dispatch of a few tokens (one launch, which needs hardly any scratch) is enough for a recorded one of the
    same shape that takes the separate launches."""
    cfg = EPConfig("graph_scratch", 12, 64, 1152, 24, 4, True)
    announce(f"recorded after a one-launch call {cfg} two_parts={two_parts}")
    world = ep.World(cfg.num_ranks)
    few = WorldHarness(cfg, world=world, num_tokens=[3] * cfg.num_ranks)
    few.load(generate(cfg, seed=90))
    few.alloc_dispatch_outputs()
    few.dispatch()
    torch.cuda.synchronize()
    assert world.get_option("last_dispatch_launches") == 1
    world.set_option("fused_small_max", 12 * 64 * 4 - 1)         # so that all the tokens take the separate launches
    data = generate(cfg, seed=91)
    h = WorldHarness(cfg, world=world, num_tokens=[5] * cfg.num_ranks if two_parts else None)
    h.load(data)
    h.alloc_dispatch_outputs(poison=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        if two_parts:
            h.dispatch(phases=1)
            h.dispatch(phases=6)
        else:
            h.dispatch()
    for _ in range(3):
        g.replay()
        few.dispatch()
        torch.cuda.synchronize()
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
        compare_dispatch(h, ref, check_poison=True)


@pytest.mark.parametrize("warm", [False, True], ids=["searched", "listed"])
def test_cast_back_of_many_experts_recorded(gpu_device, oracle, warm):
    """The work list of a cast back needs scratch; recorded without it, the kernel's blocks search for themselves."""
    R, T, H, E = 1, 8, 256, 1800
    cfg = EPConfig("graph_cast", R, T, H, E, 0, True)
    announce(f"recorded cast back {cfg} warm={warm}")
    h = WorldHarness(cfg, world=ep.World(R))
    h.alloc_dispatch_outputs(poison=False)
    h.alloc_combine_io()
    gen = torch.Generator().manual_seed(92)
    h.recv_x.copy_(torch.randint(0, 0x7f, h.recv_x.shape, generator=gen).to(torch.uint8))
    h.recv_scales_phys.copy_(torch.rand(h.recv_scales_phys.shape, generator=gen) + 0.01)
    factor = (torch.rand(E, generator=gen) + 0.5).to(gpu_device)
    torch.cuda.synchronize()
    if warm:
        h.cast_back(factor)
        torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        h.cast_back(factor)
    for i in range(3):
        h.recv_count.copy_(torch.randint(0, T + 1, h.recv_count.shape, generator=gen, dtype=torch.int32))
        want = oracle.cast_back(h.recv_x.cpu().view(torch.uint8), h.recv_scales().cpu(), h.recv_count.cpu(), factor.cpu(),
                                fill=0x5A5A)
        for call in (g.replay, lambda: h.cast_back(factor)):
            h.expert_out.view(torch.int16).fill_(0x5A5A)
            call()
            torch.cuda.synchronize()
            assert torch.equal(h.expert_out.cpu().view(torch.int16), want.view(torch.int16)), f"pass {i}"


def test_a_recorded_call_takes_the_one_launch_rather_than_fail(gpu_device, oracle):
    """The eager call's list is one that a wave counts alone, which leaves no scratch for the separate launches.  The recorded
    one has seven rounds of one list: by the measured lines the separate launches, but the shared count can take it."""
    cfg = EPConfig("graph_could", 1, 3584, 640, 8, 1, True)
    announce(f"recorded without scratch for the separate launches {cfg}")
    world = ep.World(1)
    few = WorldHarness(cfg, world=world, num_tokens=[100])
    few.load(generate(cfg, seed=94))
    few.alloc_dispatch_outputs()
    few.dispatch()
    torch.cuda.synchronize()
    assert world.get_option("last_dispatch_launches") == 1
    data = generate(cfg, seed=95)
    h = WorldHarness(cfg, world=world)
    h.load(data)
    h.alloc_dispatch_outputs(poison=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        h.dispatch()
    assert world.get_option("last_dispatch_launches") == 1
    ref = oracle.dispatch(data["x"], data["topk_idx"], [3584], 3584, 8, True)
    for _ in range(3):
        g.replay()
        few.dispatch()
        torch.cuda.synchronize()
        compare_dispatch(h, ref, check_poison=True)
    h.dispatch()                                    # an eager call makes room for the separate launches and takes them
    torch.cuda.synchronize()
    assert world.get_option("last_dispatch_launches") > 1
    compare_dispatch(h, ref, check_poison=True)
