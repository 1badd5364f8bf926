"""Combine of a handle that is not the last dispatch's, looked up by the reduce kernels themselves (one launch) or
turned into routes by a resolve launch first: both against the oracle, bit for bit, at every share of a wave that a
selection can have (top-k brackets), with ranges longer than a wave scans at a time, ranks without tokens, repeated
experts, masked selections, an inactive rank, an empty and a malformed range, and the packed combine."""
import pytest
import torch

from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, run_dispatch

pytestmark = pytest.mark.gpu

CASES = [
    EPConfig("k1", 3, 96, 256, 3, 1, False),                # one selection per wave; a range is all 96 tokens at most
    EPConfig("k2_one_expert", 1, 256, 256, 2, 2, False),    # ranges of 256: two rounds of the scan
    EPConfig("k3", 4, 33, 640, 8, 3, True),
    EPConfig("k6", 2, 40, 1152, 12, 6, True),
    EPConfig("k8_hot", 4, 129, 512, 16, 8, False, routing="zipf"),
    EPConfig("k11", 2, 30, 384, 22, 11, False, masked_fraction=0.2),
    EPConfig("k16_hot", 2, 64, 256, 16, 16, True),          # every token names every expert
]


@pytest.mark.parametrize("cfg", CASES, ids=[c.name for c in CASES])
@pytest.mark.parametrize("uniform", [1, 0], ids=["spaced", "table"])
def test_searched_and_resolved_handles_match_oracle(gpu_device, oracle, cfg, uniform):
    R, T, E, K, L = cfg.num_ranks, cfg.tokens_per_rank, cfg.num_experts, cfg.num_topk, cfg.num_local_experts
    nt = [max(0, T - r * 11) for r in range(R)]
    if R > 2:
        nt[1] = 0
    announce(f"combine by search and by resolve {cfg} nt={nt} uniform={uniform}")
    data = generate(cfg, seed=71)
    if K > 1:
        data["topk_idx"][0, ::4, K - 1] = data["topk_idx"][0, ::4, 0]     # a repeated expert: its last row counts twice
    h = run_dispatch(cfg, data, num_tokens=nt, poison=True, options={"combine_direct": 0, "uniform": uniform})
    factor = torch.arange(E).float() * 0.1 + 0.5
    h.alloc_combine_io()
    h.cast_back(factor)
    torch.cuda.synchronize()
    active = torch.ones(R, R, dtype=torch.int32)
    if R > 1:
        active[0, R - 1] = 0
    h.active_ranks.copy_(active.to(h.active_ranks.dtype))
    # one range emptied, one that does not fit its block
    lr = h.layout_range.cpu()
    lr[0, 0, 0] = 0
    if R * L > 1:
        lr[R - 1, L - 1, 0] = (R * T << 32) | 1
    h.layout_range.copy_(lr)
    lr[R - 1, L - 1, 0] = 0                                                # which has no rows, as an empty one
    # rows that repeated experts got beyond a block's capacity are nobody's: the oracle's ranges hold none either
    want = oracle.combine(h.expert_out.cpu(), data["topk_idx"], data["topk_weights"], h.src_info.cpu(), lr, nt,
                          cfg.max_tokens, E, active=active)
    for packed in (False, True):
        for tokens in (256, 0):
            h.world.set_option("combine_search_tokens", tokens)
            h.combined.fill_(7.0)
            if packed:
                h.combine_packed(factor)
            else:
                h.combine()
            torch.cuda.synchronize()
            launches = h.world.get_option("last_combine_launches")
            assert launches == 1 if tokens else launches >= 2
            for r, n in enumerate(nt):
                assert torch.equal(h.combined[r, :n].cpu().view(torch.int16), want[r, :n].view(torch.int16)), \
                    f"rank {r} packed={packed} search={tokens}"
                assert bool((h.combined[r, n:] == 7.0).all())


def test_the_search_rule(gpu_device):
    announce("combine: the rule for searched handles")
    for T, one in ((256, True), (257, False)):
        cfg = EPConfig("rule", 2, T, 128, 4, 2, False)
        h = run_dispatch(cfg, generate(cfg, seed=72), poison=False, options={"combine_direct": 0})
        h.alloc_combine_io()
        h.cast_back(None)
        h.combine()
        torch.cuda.synchronize()
        assert (h.world.get_option("last_combine_launches") == 1) == one


def test_the_search_rule_by_top_k(gpu_device):
    announce("combine: the rule for searched handles, by selections a token")
    for K, T, one in ((4, 256, True), (5, 96, True), (5, 97, False), (7, 97, False), (8, 160, True), (8, 161, False),
                      (9, 64, True), (9, 65, False), (16, 64, True), (16, 65, False)):
        cfg = EPConfig("rule", 2, T, 128, 16, K, False)
        h = run_dispatch(cfg, generate(cfg, seed=73), poison=False, options={"combine_direct": 0})
        h.alloc_combine_io()
        h.cast_back(None)
        h.combine()
        torch.cuda.synchronize()
        assert (h.world.get_option("last_combine_launches") == 1) == one, (K, T)


@pytest.mark.parametrize("tokens", [256, 0], ids=["searched", "resolved"])
def test_ranges_longer_than_the_tokens_combined(gpu_device, oracle, tokens):
    """A handle of many tokens, of which a few are combined; and ranges that repeated experts make longer than that."""
    cfg = EPConfig("long_ranges", 2, 700, 256, 4, 2, True)
    announce(f"combine of a few tokens of a long handle, search={tokens}")
    data = generate(cfg, seed=74)
    data["topk_idx"][1, ::2, 1] = data["topk_idx"][1, ::2, 0]
    h = run_dispatch(cfg, data, poison=True, options={"combine_search_tokens": tokens})
    factor = torch.arange(4).float() * 0.1 + 0.5
    h.alloc_combine_io()
    h.cast_back(factor)
    torch.cuda.synchronize()
    assert int((h.layout_range.cpu() & 0xffffffff).max()) > 300
    h.num_tokens = [5, 256]
    want = oracle.combine(h.expert_out.cpu(), data["topk_idx"], data["topk_weights"], h.src_info.cpu(),
                          h.layout_range.cpu(), h.num_tokens, cfg.max_tokens, 4)
    for packed in (False, True):
        h.combined.fill_(7.0)
        if packed:
            h.combine_packed(factor)
        else:
            h.combine()
        torch.cuda.synchronize()
        assert (h.world.get_option("last_combine_launches") == 1) == (tokens > 0)
        for r, n in enumerate(h.num_tokens):
            assert torch.equal(h.combined[r, :n].cpu().view(torch.int16), want[r, :n].view(torch.int16)), f"rank {r}"
            assert bool((h.combined[r, n:] == 7.0).all())
