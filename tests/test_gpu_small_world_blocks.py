"""The one-launch dispatch with several tokens a block, which share one walk through the index lists: every number of
tokens a block can have (eight, four and two, with eight or six waves), token counts that leave the last block part empty,
repeated experts within a token and across a block's tokens, numbers no expert has, ranks without tokens, thousands of
experts, top-k from 1 to 16; and the size rule on either side of its lines.  Bit for bit against the oracle,
with the combine that reads where the selections went."""
import pytest
import torch

from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, compare_dispatch, run_dispatch

pytestmark = pytest.mark.gpu

CASES = [
    EPConfig("eight_k8", 1, 600, 1024, 16, 8, True),                       # 4800 selections, one list
    EPConfig("eight_k16", 2, 150, 640, 32, 16, True, routing="zipf"),      # 128 entries in a block
    EPConfig("eight_k16_bf16", 1, 512, 640, 32, 16, False),                # 8192, by the cap that the test sets
    EPConfig("eight_k1", 12, 64, 1024, 24, 1, True, routing="zipf"),       # 64 lanes on a selection
    EPConfig("eight_k2", 1, 2040, 1024, 16, 2, True, masked_fraction=0.1),
    EPConfig("four_k9", 12, 72, 1920, 36, 9, True, masked_fraction=0.2),   # 7776
    EPConfig("four_k3", 12, 150, 2048, 24, 3, False, routing="zipf"),      # 5400
    EPConfig("two_of_three", 2, 300, 2944, 18, 8, True),                   # six waves
    EPConfig("two_of_four", 8, 80, 4096, 64, 8, False),                    # 5120
    EPConfig("few_selections", 12, 70, 1152, 108, 5, True),                # 4200 as listed, fewer when ragged
    EPConfig("lists_of_many_ranks", 24, 20, 3072, 48, 8, True),            # 3840
    EPConfig("most_experts", 16, 40, 640, 3584, 8, False),                 # 5120, and nearly all the experts that are taken
]
BLOCK = {"eight": 8, "four": 4, "two": 2, "few": 4, "lists": 2, "most": 8}    # tokens of a block, by the name's first word


@pytest.mark.parametrize("cfg", CASES, ids=[c.name for c in CASES])
@pytest.mark.parametrize("is_ragged", [False, True], ids=["full", "ragged"])
def test_blocks_of_several_tokens_match_oracle(gpu_device, oracle, cfg, is_ragged):
    R, T, E, K = cfg.num_ranks, cfg.tokens_per_rank, cfg.num_experts, cfg.num_topk
    nt = [T - r % 5 for r in range(R)] if is_ragged else None
    if is_ragged and R > 2:
        nt[1] = 0
    announce(f"one-launch dispatch, several tokens a block {cfg} nt={nt}")
    data = generate(cfg, seed=83)
    if K > 1:
        data["topk_idx"][0, 3:T:4, K - 1] = data["topk_idx"][0, 3:T:4, 0]  # twice in a token
    data["topk_idx"][0, 1:8, 0] = data["topk_idx"][0, 0, 0]                # and by every token of the first blocks
    if is_ragged:
        data["topk_idx"][0, 5, K // 2] = 2 ** 32 + 1
    # (K a power of two and not)
    options = {"fused_small_max": 8192} if cfg.name == "eight_k16_bf16" else {}
    h = run_dispatch(cfg, data, num_tokens=nt, poison=True, options=options)
    assert h.world.get_option("last_dispatch_launches") == 1
    assert h.world.get_option("last_dispatch_block_tokens") == BLOCK[cfg.name.split("_")[0]]
    ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, E, cfg.use_fp8)
    compare_dispatch(h, ref, check_poison=True)
    h.alloc_combine_io()
    h.cast_back()                       # (a repeated expert's rows are equal: any of them may count)
    h.combine()
    torch.cuda.synchronize()
    want = oracle.combine(h.expert_out.cpu(), data["topk_idx"], data["topk_weights"], ref["src_info"], ref["layout_range"],
                          h.num_tokens, cfg.max_tokens, E)
    for r, n in enumerate(h.num_tokens):
        assert torch.equal(h.combined[r, :n].cpu().view(torch.int16), want[r, :n].view(torch.int16)), r


def test_size_rule_of_shared_blocks(gpu_device, oracle):
    announce("one-launch dispatch, several tokens a block: the size rule")
    base = EPConfig("base", 1, 640, 1024, 16, 8, True)
    from dataclasses import replace
    cases = [(base, {}, 1, 8),                                                    # 5120 selections
             (base, {"fused_shared_max": 5119}, 2, 0),
             (base, {"fused_shared_max": 5120}, 1, 8),
             (base, {"fused_small_max": 5119}, 2, 0),                             # a cap that a program sets
             (base, {"fused_small": 0}, 2, 0),
             (replace(base, num_topk=2, tokens_per_rank=2100), {}, 2, 0),         # top-2
             (replace(base, hidden=512), {}, 3, 0),                               # half a slab
             (replace(base, hidden=4224), {}, 2, 0),                              # one token a block
             (replace(base, hidden=4096, tokens_per_rank=1228, num_topk=4), {}, 1, 2),   # 1228 x 10 rounds, 6144 x 2 at most
             (replace(base, hidden=4096, tokens_per_rank=1232, num_topk=4), {}, 2, 0),   # 1232 x 10
             (replace(base, hidden=2048, num_ranks=32, tokens_per_rank=22, num_experts=32), {}, 1, 4),   # 32 lists, 704 x 32 rounds
             (replace(base, num_ranks=32, tokens_per_rank=22, num_experts=32), {}, 2, 0),    # ... of short rows
             (replace(base, num_ranks=2, tokens_per_rank=1028, num_experts=16), {}, 2, 0),   # 16448 selections
             (replace(base, tokens_per_rank=64), {}, 1, 1)]                       # one list: a token a block
    for cfg, options, launches, tokens in cases:
        data = generate(cfg, seed=84)
        h = run_dispatch(cfg, data, poison=True, options=options)
        assert h.world.get_option("last_dispatch_launches") == launches, (cfg, options)
        assert h.world.get_option("last_dispatch_block_tokens") == tokens, (cfg, options)
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, True)
        compare_dispatch(h, ref, check_poison=True)


def test_recorded_shared_blocks_replay(gpu_device, oracle):
    """The one launch for thousands of selections in a graph: replays on fresh inputs, with eager calls in between."""
    from mooncake_amd import ep
    from mooncake_amd.harness import WorldHarness

    cfg = EPConfig("recorded", 2, 300, 2048, 16, 8, True)
    announce(f"one-launch dispatch, several tokens a block, recorded {cfg}")
    h = WorldHarness(cfg, world=ep.World(2))
    h.load(generate(cfg, seed=85))
    h.alloc_dispatch_outputs()
    h.alloc_combine_io()
    h.expert_out.normal_()
    h.dispatch()
    h.combine()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        h.dispatch()
        h.combine()
    assert h.world.get_option("last_dispatch_launches") == 1
    assert h.world.get_option("last_dispatch_block_tokens") == 4
    for seed in (86, 87, 88):
        data = generate(cfg, seed=seed)
        h.x.copy_(data["x"])
        h.topk_idx.copy_(data["topk_idx"])
        h.topk_weights.copy_(data["topk_weights"])
        g.replay()
        torch.cuda.synchronize()
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, True)
        compare_dispatch(h, ref, check_poison=False)
        want = oracle.combine(h.expert_out.cpu(), data["topk_idx"], data["topk_weights"], ref["src_info"],
                              ref["layout_range"], h.num_tokens, cfg.max_tokens, cfg.num_experts)
        assert torch.equal(h.combined.cpu().view(torch.int16), want.view(torch.int16)), seed
        h.dispatch()
        torch.cuda.synchronize()
