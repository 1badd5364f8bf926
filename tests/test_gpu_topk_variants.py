"""Combine and packed combine at every top-k from 1 to 16: the kernels have variants for some numbers of rows (each one of
them for fp8 payloads) and pad to the next one in between, and the packed combine of an fp8 payload fetches a slab's scales
with the lanes of all selections together.  Rows from the dispatch, from the handle and from routes; a hidden size whose last
slab holds one scale group; masked tokens and an inactive rank.  Bit for bit against the oracle."""
import pytest
import torch

from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce, run_dispatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_fp8", [True, False], ids=["fp8", "bf16"])
@pytest.mark.parametrize("topk", range(1, 17))
def test_every_topk_matches_oracle(gpu_device, oracle, topk, use_fp8):
    cfg = EPConfig(f"k{topk}", 2, 22, 1152, 32, topk, use_fp8, masked_fraction=0.1)
    announce(f"combine variants {cfg}")
    data = generate(cfg, seed=90 + topk)
    nt = [22, 17]
    h = run_dispatch(cfg, data, num_tokens=nt, poison=True)
    factor = torch.arange(cfg.num_experts).float() * 0.1 + 0.5
    h.alloc_combine_io()
    active = torch.tensor([[1, 0], [1, 1]], dtype=torch.int32)
    h.active_ranks.copy_(active.to(h.active_ranks.dtype))
    ref = oracle.dispatch(data["x"], data["topk_idx"], nt, cfg.max_tokens, cfg.num_experts, use_fp8)
    for f in (factor, None):
        h.cast_back(f)
        rows = oracle.cast_back(ref["recv_x"], ref["scales"] if use_fp8 else None, ref["recv_count"], f)
        want = oracle.combine(rows, data["topk_idx"], data["topk_weights"], ref["src_info"], ref["layout_range"], nt,
                              cfg.max_tokens, cfg.num_experts, active=active)
        for direct, tokens in ((1, 256), (0, 256), (0, 0)):
            h.world.set_option("combine_direct", direct)
            h.world.set_option("combine_search_tokens", tokens)
            for call in (h.combine, lambda: h.combine_packed(f)):
                h.combined.fill_(7.0)
                call()
                torch.cuda.synchronize()
                got = h.combined.cpu()
                for r, n in enumerate(nt):
                    assert torch.equal(got[r, :n].view(torch.int16), want[r, :n].view(torch.int16)), (direct, tokens, r)
                    assert bool((got[r, n:] == 7.0).all()), "rows beyond num_tokens written"


def test_a_last_slab_of_few_elements_takes_no_longer(gpu_device):
    """Packed combine of rows whose last slab has one scale group, against rows that are longer by three: the arithmetic is
    done by all lanes of a wave.  (Under the mask of the lanes inside the row, eight of 64, it took 2.2 times as long.)"""
    announce("packed combine, a last slab of one scale group")
    best = {}
    for hidden in (1152, 1536):
        cfg = EPConfig("slab", 1, 64, hidden, 16, 16, True)
        h = run_dispatch(cfg, generate(cfg, seed=120), poison=False)
        h.alloc_combine_io()
        factor = torch.ones(cfg.num_experts)
        h.combine_packed(factor)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            h.dispatch()
            for _ in range(20):
                h.combine_packed(h._factor)
        best[hidden] = float("inf")
        for _ in range(20):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            g.replay()
            end.record()
            torch.cuda.synchronize()
            best[hidden] = min(best[hidden], start.elapsed_time(end))
    assert best[1152] < 1.5 * best[1536], best
