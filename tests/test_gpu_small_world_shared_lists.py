"""The one-launch dispatch where the waves of a block share the index lists out: several slabs per token (so several
waves and more than 8 ranks), lists around the 512-entry rounds the waves take in turn, more slabs than a block has
waves, more experts than its histogram holds at a time.  Whole numbers and bytes: everything equals the oracle's."""
import pytest

from mooncake_amd.workloads import EPConfig, generate
from tests import gpu_util
from tests.gpu_util import announce, compare_dispatch, run_dispatch

pytestmark = pytest.mark.gpu

CASES = [
    EPConfig("ranks_12_two_slabs", 12, 68, 1152, 108, 5, True),      # 12 lists of 340 entries on four waves
    EPConfig("ranks_32_four_waves", 32, 8, 640, 32, 3, False),       # the most ranks there are, on the fewest waves
    EPConfig("ranks_32_eight_slabs", 32, 16, 7424, 64, 8, True),     # the most ranks there are
    EPConfig("rounds_512_513", 3, 171, 1152, 24, 3, False),          # 513 entries: a round and one entry
    EPConfig("rounds_6_of_512", 1, 384, 4096, 64, 8, True),          # one list, six whole rounds
    EPConfig("slabs_9", 2, 12, 9216, 16, 4, True),                   # a slab more than a block has waves
    EPConfig("slabs_18_bf16", 2, 5, 17536, 16, 4, False),
    EPConfig("experts_4096", 4, 16, 1152, 4096, 8, True),            # a whole histogram, and one with a remainder
    EPConfig("experts_8200", 4, 16, 1152, 8200, 8, False),
    EPConfig("hot", 8, 64, 4096, 64, 6, True, routing="zipf", masked_fraction=0.2),
]


@pytest.mark.parametrize("cfg", CASES, ids=[c.name for c in CASES])
@pytest.mark.parametrize("is_ragged", [False, True], ids=["full", "ragged"])
def test_shared_lists_match_oracle(gpu_device, oracle, cfg, is_ragged):
    T = cfg.tokens_per_rank
    nt = [T - r * 7 % (T + 1) for r in range(cfg.num_ranks)] if is_ragged else None
    announce(f"one-launch dispatch, shared lists {cfg} ragged={nt}")
    data = generate(cfg, seed=61)
    if is_ragged:
        data["topk_idx"][0, ::5, -1] = data["topk_idx"][0, ::5, 0]    # repeated experts
        data["topk_idx"][-1, 0, 0] = 2 ** 32 + 1                      # and a number no expert has
    gpu_util.DEFAULT_OPTIONS["fused_small_rounds"] = 1 << 20
    try:
        h = run_dispatch(cfg, data, num_tokens=nt, poison=True)
    finally:
        gpu_util.DEFAULT_OPTIONS.pop("fused_small_rounds", None)
    assert h.world.get_option("last_dispatch_launches") == 1
    ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
    compare_dispatch(h, ref, check_poison=True)


def test_size_rule_per_wave(gpu_device, oracle):
    """Up to six rounds a wave for fp8 and four for bf16: four waves up to hidden 4096, a wave per 1024 elements above."""
    announce("one-launch dispatch, the size rule per wave")
    for cfg, one in ((EPConfig("fp8_24_lists", 24, 4, 1152, 24, 2, True), True),
                     (EPConfig("fp8_25_lists", 25, 4, 1152, 25, 2, True), False),
                     (EPConfig("bf16_16_lists", 16, 4, 640, 16, 2, False), True),
                     (EPConfig("bf16_17_lists", 17, 4, 640, 17, 2, False), False),
                     (EPConfig("fp8_30_lists_5_waves", 30, 4, 4224, 30, 2, True), True),
                     (EPConfig("fp8_31_lists_5_waves", 31, 4, 4224, 31, 2, True), False)):
        data = generate(cfg, seed=62)
        h = run_dispatch(cfg, data, poison=True)
        assert (h.world.get_option("last_dispatch_launches") == 1) == one, cfg.name
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
        compare_dispatch(h, ref, check_poison=True)


def test_what_no_path_but_this_could_take(gpu_device):
    """More experts than the count kernel's LDS holds: taken while one wave could count the lists, refused beyond."""
    announce("one-launch dispatch, more experts than the other path takes")
    cfg = EPConfig("few_lists", 4, 16, 1152, 8200, 8, True)
    h = run_dispatch(cfg, generate(cfg, seed=63), poison=False)
    assert h.world.get_option("last_dispatch_launches") == 1
    cfg = EPConfig("many_lists", 10, 4, 1152, 8200, 8, True)
    with pytest.raises(RuntimeError):
        run_dispatch(cfg, generate(cfg, seed=63), poison=False)


def test_size_rule_prices_the_rounds_that_are_walked(gpu_device, oracle):
    """A wave goes through as many rounds of every rank as the longest list has, and every token goes through them: very
    uneven lists and thousands of tokens with one or two selections each take the separate launches."""
    announce("one-launch dispatch, the size rule for uneven lists and many tokens")
    cases = [
        (EPConfig("8_ranks_one_long", 8, 440, 1024, 64, 8, True), [440] + [10] * 7, False),     # 8 x 7 rounds on 4 waves
        (EPConfig("12_ranks_last_long", 12, 256, 1024, 48, 8, True), [8] * 11 + [256], False),
        (EPConfig("4_ranks_one_long", 4, 320, 1024, 64, 8, True), [320, 8, 8, 8], True),        # 4 x 5 on 4 waves
        (EPConfig("top1_4096", 1, 4096, 640, 8, 1, True), None, False),                         # 32768 rounds in all
        (EPConfig("top2_2048", 1, 2048, 640, 8, 2, True), None, True),                          # 16384
        (EPConfig("top2_2048_bf16", 1, 2048, 640, 8, 2, False), None, False),
        (EPConfig("top4_1024_bf16", 1, 1024, 640, 8, 4, False), None, True),                    # 8192
    ]
    for cfg, nt, one in cases:
        data = generate(cfg, seed=67)
        h = run_dispatch(cfg, data, num_tokens=nt, poison=True)
        assert (h.world.get_option("last_dispatch_launches") == 1) == one, cfg.name
        ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
        compare_dispatch(h, ref, check_poison=True)
