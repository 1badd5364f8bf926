"""Write-through payload stores of the pack kernels (`pack_nt` bit 2): buffer stores bounded by the row, so the rows
to check are the ones whose last 1024-element slab is partly, or hardly, there, and the largest the path takes."""
import pytest

from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, compare_dispatch, run_dispatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_fp8", [True, False], ids=["fp8", "bf16"])
@pytest.mark.parametrize("hidden", [128, 1024, 1152, 2560, 32768])
@pytest.mark.parametrize("nt", [4, 5])
def test_write_through_rows_match_oracle(gpu_device, oracle, nt, hidden, use_fp8):
    cfg = EPConfig("through", 4, 9, hidden, 12, 3, use_fp8, masked_fraction=0.2)
    announce(f"write-through stores pack_nt={nt} {cfg}")
    data = generate(cfg, seed=5)
    h = run_dispatch(cfg, data, num_tokens=[9, 0, 4, 9], poison=True, options={"fused_small": 0, "pack_nt": nt})
    ref = oracle.dispatch(data["x"], data["topk_idx"], h.num_tokens, cfg.max_tokens, cfg.num_experts, use_fp8)
    compare_dispatch(h, ref, check_poison=True)
