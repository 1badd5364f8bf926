"""Edges of the layout kernels against the oracle, bit for bit: worlds with as many units of 256 selections as a wave of
the prefix pass loads at a time (512), one more and one fewer, and scale counts per row around the 16 that a wave of the
scale transposition takes (whole, with a remainder of whole and of partial 16-byte pieces)."""
import pytest

from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, compare_dispatch, run_dispatch

pytestmark = pytest.mark.gpu


def check(oracle, cfg, nt=None, **options):
    data = generate(cfg, seed=81)
    h = run_dispatch(cfg, data, num_tokens=nt, poison=True, options={"fused_small": 0, **options})
    ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, cfg.use_fp8)
    compare_dispatch(h, ref, check_poison=True)


@pytest.mark.parametrize("units", [511, 512, 513])
def test_prefix_over_many_units(gpu_device, oracle, units):
    announce(f"prefix pass over {units} units")
    check(oracle, EPConfig("units", 1, units * 32 - 3, 128, 8, 8, False))


@pytest.mark.parametrize("units,experts", [(64, 1023), (65, 1023), (65, 1024), (130, 1024)])
def test_prefix_pass_by_units_and_experts(gpu_device, oracle, units, experts):
    """Both sides of the line between one and eight pieces of the counts in flight."""
    announce(f"prefix pass over {units} units of {experts} experts")
    check(oracle, EPConfig("units", 1, units * 64 - 3, 128, experts, 4, False), routing_sum=0)


@pytest.mark.parametrize("groups", [15, 16, 17, 20, 32, 36])
def test_scale_transposition_parts(gpu_device, oracle, groups):
    announce(f"scale transposition of {groups} groups")
    check(oracle, EPConfig("groups", 4, 70, groups * 128, 8, 3, True), nt=[70, 3, 0, 66])
