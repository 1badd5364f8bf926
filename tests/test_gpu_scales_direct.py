"""fp8 dispatch with few scales: the pack kernel stores them in their columns by itself, without the transposing launch.
Either side of the line (by size, by hidden, by option and by phases), with the summed and the table routing plan, both
statements of the scale arithmetic, odd hidden sizes, ragged ranks, masked tokens, repeated experts, and ranks that take no
part; a later call of the last phase alone still finds what it needs.  Bit for bit against the oracle."""
import pytest
import torch

from mooncake_amd import _lib
from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, compare_dispatch, run_dispatch

pytestmark = pytest.mark.gpu

# config, launches of the dispatch with one pack launch for the scales too
CASES = [
    (EPConfig("h640", 3, 480, 640, 12, 3, True, masked_fraction=0.1), 2),          # 4257 selections, 5 groups
    (EPConfig("h1152_k9", 4, 128, 1152, 32, 9, True), 2),                          # the last slab holds one group
    (EPConfig("one_rank", 1, 1024, 1024, 16, 5, True, routing="zipf"), 2),
    (EPConfig("line", 1, 4096, 1280, 8, 8, True), 2),                              # 320 x 1024 scales exactly
    (EPConfig("beyond_line", 1, 4100, 1280, 8, 8, True), 3),
    (EPConfig("half_slab", 2, 600, 512, 8, 4, True), 3),
]


@pytest.mark.parametrize("cfg,launches", CASES, ids=[c.name for c, _ in CASES])
@pytest.mark.parametrize("plan", [1, 0], ids=["summed", "table"])
@pytest.mark.parametrize("arith", [0, 1], ids=["torch", "kernel"])
def test_scales_in_place(gpu_device, oracle, cfg, launches, plan, arith):
    R, T, K = cfg.num_ranks, cfg.tokens_per_rank, cfg.num_topk
    nt = [T - 7 * r for r in range(R)]
    announce(f"scales in place {cfg} plan={plan} arith={arith}")
    data = generate(cfg, seed=17)
    if K > 1:
        data["topk_idx"][0, ::5, K - 1] = data["topk_idx"][0, ::5, 0]     # a repeated expert has a row per occurrence
    h = run_dispatch(cfg, data, num_tokens=nt, poison=True, options={"routing_sum": plan, "fp8_arith": arith, "fused_small": 0})
    oracle.set_fp8_arith(arith)
    try:
        ref = oracle.dispatch(data["x"], data["topk_idx"], nt, cfg.max_tokens, cfg.num_experts, True)
    finally:
        oracle.set_fp8_arith(0)
    assert h.world.get_option("last_dispatch_launches") >= launches        # (a table plan has a prefix launch besides)
    assert plan == 0 or h.world.get_option("last_dispatch_launches") == launches
    compare_dispatch(h, ref, check_poison=True)
    # the last phase by itself, over scales that were overwritten: it reads what the data phase staged
    h.recv_scales_phys.fill_(float("nan"))
    h.dispatch(phases=_lib.PHASE_FINISH)
    torch.cuda.synchronize()
    compare_dispatch(h, ref, check_poison=True)
    # and all phases apart: the scales are there after the last one, not before
    h.recv_scales_phys.fill_(float("nan"))
    h.dispatch(phases=_lib.PHASE_LAYOUT | _lib.PHASE_DATA)
    torch.cuda.synchronize()
    assert bool(torch.isnan(h.recv_scales_phys).all())
    h.dispatch(phases=_lib.PHASE_FINISH)
    torch.cuda.synchronize()
    compare_dispatch(h, ref, check_poison=True)


@pytest.mark.parametrize("noalloc", [False, True])
def test_scales_in_place_of_a_silent_rank_and_by_option(gpu_device, oracle, noalloc):
    cfg = EPConfig("silent", 3, 800, 640, 12, 3, True)
    data = generate(cfg, seed=18)
    got = []
    for direct in (1, 0):
        announce(f"scales in place: a silent rank, noalloc={noalloc} direct={direct}")
        h = run_dispatch(cfg, data, poison=True, present=[1, 0, 1], options={"scales_direct": direct, "fused_small": 0})
        if noalloc:
            h.recv_scales_phys.fill_(float("nan"))
            h.dispatch(present=[1, 0, 1], noalloc=True)
            torch.cuda.synchronize()
        assert h.world.get_option("last_dispatch_launches") == 3 - direct
        got.append((h.recv_count.cpu(), h.recv_x.cpu(), h.recv_scales_phys.view(torch.int32).cpu()))
    assert all(torch.equal(a, b) for a, b in zip(*got))
