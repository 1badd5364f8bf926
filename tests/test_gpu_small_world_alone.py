"""The one-launch dispatch whose waves count by themselves (top-1 and top-2 worlds, lists of a single round of 512
entries): lists around the 128-entry steps and the rounds of its counting loop, lists that start in the middle of a
16-byte unit, the edges of what is taken by it rather than by the shared count, payloads on both sides of the size from
which rows are written through the L2.  Whole numbers and bytes: everything equals the oracle's."""
import pytest

from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, compare_dispatch, run_dispatch

pytestmark = pytest.mark.gpu

CASES = [
    EPConfig("one_token", 1, 4, 128, 1, 1, True),
    EPConfig("one_round", 1, 512, 1152, 16, 1, False),
    EPConfig("one_round_and_one", 1, 513, 1152, 16, 1, False),
    EPConfig("odd_lists", 4, 257, 640, 8, 1, True),                     # every other rank's list at an odd place
    EPConfig("odd_lists_2048", 2, 1023, 256, 4, 1, False),
    EPConfig("six_rounds_hot", 1, 1536, 1024, 8, 2, True, routing="zipf", masked_fraction=0.1),
    EPConfig("shared_below_256_entries", 2, 127, 640, 4, 2, False),
    EPConfig("alone_from_256_entries", 2, 128, 640, 4, 2, False),
    EPConfig("top4_one_round", 1, 128, 2048, 64, 4, False),
    EPConfig("top4_a_round_and_four", 1, 129, 2048, 64, 4, False),
    EPConfig("top3", 1, 60, 4224, 12, 3, True),
    EPConfig("top8_bf16", 1, 37, 3072, 64, 8, False),
    EPConfig("top8_five_slabs", 1, 64, 4224, 256, 8, True),             # 2.2 MB: left to the L2
    EPConfig("top16_seven_slabs", 1, 32, 7168, 16, 16, True),
    EPConfig("top11_bf16", 1, 46, 7168, 64, 11, False),
    EPConfig("top5_written_through", 1, 100, 9216, 256, 5, True),       # 4.6 MB
    EPConfig("top2_written_through", 8, 300, 1024, 8, 2, False),
]


@pytest.mark.parametrize("cfg", CASES, ids=[c.name for c in CASES])
@pytest.mark.parametrize("is_ragged", [False, True], ids=["full", "ragged"])
def test_alone_matches_oracle(gpu_device, oracle, cfg, is_ragged):
    T, R = cfg.tokens_per_rank, cfg.num_ranks
    nt = [T - r * 7 % (T + 1) for r in range(R)] if is_ragged else None
    announce(f"one-launch dispatch, every wave alone {cfg} ragged={nt}")
    data = generate(cfg, seed=64)
    if is_ragged:
        data["topk_idx"][0, ::5, -1] = data["topk_idx"][0, ::5, 0]    # repeated experts
        data["topk_idx"][-1, 0, 0] = 2 ** 32 + 1                      # and a number no expert has
    h = run_dispatch(cfg, data, num_tokens=nt, poison=True, options={"fused_small_rounds": 16, "fused_small_max": 1 << 13})
    assert h.world.get_option("last_dispatch_launches") == 1
    ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
    compare_dispatch(h, ref, check_poison=True)


@pytest.mark.parametrize("arith", [0, 1], ids=["torch_arith", "kernel_arith"])
def test_fp8_arithmetic_options(gpu_device, oracle, arith):
    cfg = EPConfig("arith", 1, 36, 2560, 16, 3, True, outlier_fraction=0.1)
    announce(f"one-launch dispatch, every wave alone, fp8_arith={arith}")
    data = generate(cfg, seed=65)
    h = run_dispatch(cfg, data, poison=True, options={"fp8_arith": arith})
    assert h.world.get_option("last_dispatch_launches") == 1
    oracle.set_fp8_arith(arith)
    try:
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, True)
    finally:
        oracle.set_fp8_arith(0)
    compare_dispatch(h, ref, check_poison=True)


def test_silent_rank_and_rank_that_receives_nothing(gpu_device, oracle):
    cfg = EPConfig("silent", 4, 300, 640, 8, 1, True)
    announce(f"one-launch dispatch, every wave alone, silent rank {cfg}")
    data = generate(cfg, seed=66)
    present = [1, 0, 1, 1]
    h = run_dispatch(cfg, data, poison=True, present=present)
    assert h.world.get_option("last_dispatch_launches") == 1
    ref = oracle.dispatch(data["x"], data["topk_idx"], [300, 0, 300, 300], cfg.max_tokens, cfg.num_experts, True)
    for r in (0, 2, 3):
        assert h.recv_count[r].tolist() == ref["recv_count"][r].tolist()
        assert h.layout_range[r].tolist() == ref["layout_range"][r].tolist()
    assert bool((h.recv_count[1] == -7).all()) and bool((h.src_info[1] == -7).all())
