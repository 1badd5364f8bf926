"""The cast-back kernel's search for the rows of its 16-row chunks, at its edges, against the oracle bit for bit:
counts around the chunk size, experts without rows, one to sixteen experts per searching thread, scales whose columns are
no multiple of four rows, more ranks than travel in kernel arguments, worlds
of so many experts that the chunks come from a work list, unevenly spaced count tensors, an absent rank."""
import pytest
import torch

from mooncake_amd import ep
from mooncake_amd.harness import WorldHarness
from mooncake_amd.workloads import EPConfig
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu

FILL = 0x5A5A
EDGES = [0, 1, 15, 16, 17, 0, 0, 31, 32, 33, 4, 5]


@pytest.mark.parametrize("use_fp8", [True, False], ids=["fp8", "bf16"])
@pytest.mark.parametrize("shape", [
    # ranks, tokens, hidden, experts, absent rank
    (1, 33, 1152, 1, None), (1, 35, 128, 12, None), (3, 12, 1024, 255, 1), (4, 9, 256, 260, None), (2, 17, 2176, 514, 0),
    (3, 11, 128, 1281, None), (2, 20, 128, 2050, None), (4, 9, 256, 4096, 2),
    (33, 3, 1152, 1056, 5), (32, 2, 128, 64, 7), (33, 1, 256, 99, 32),
], ids=lambda s: "x".join(str(v) for v in s))
def test_chunk_edges(gpu_device, oracle, shape, use_fp8):
    R, T, H, E, absent = shape
    cfg = EPConfig("chunks", R, T, H, E, 0, use_fp8)
    announce(f"cast-back chunks {shape} fp8={use_fp8}")
    h = WorldHarness(cfg, world=ep.World(R))
    h.alloc_dispatch_outputs(poison=False)
    h.alloc_combine_io()
    L, RM = E // R, R * T
    gen = torch.Generator().manual_seed(E)
    if use_fp8:
        h.recv_x.copy_(torch.randint(0, 0x7f, h.recv_x.shape, generator=gen).to(torch.uint8))
        h.recv_scales_phys.copy_(torch.rand(h.recv_scales_phys.shape, generator=gen) + 0.01)
    else:
        h.recv_x.view(torch.bfloat16).copy_(torch.randn(h.recv_x.shape, generator=gen))
    counts = torch.tensor([min(RM, EDGES[(e * 7 + e // 12) % len(EDGES)]) for e in range(E)], dtype=torch.int32)
    h.recv_count.copy_(counts.view(R, L))
    factor = torch.rand(E, generator=gen) + 0.5
    scales = h.recv_scales().cpu() if use_fp8 else None
    recv = h.recv_x.cpu().view(torch.uint8 if use_fp8 else torch.bfloat16)
    want = oracle.cast_back(recv, scales, h.recv_count.cpu(), factor, fill=FILL)
    present = None if absent is None else [int(r != absent) for r in range(R)]
    # evenly spaced counts, then each rank's in a tensor of its own
    spread = [h.recv_count[r].clone() for r in range(R)]
    spread.reverse()
    for r in range(R):
        spread[r].copy_(h.recv_count[r])
    for count_ptrs in (None, [t.data_ptr() for t in spread]):
        h.expert_out.view(torch.int16).fill_(FILL)
        if count_ptrs is None:
            h.cast_back(factor, present=present)
        else:
            h.world.cast_back(h._ptrs(h.recv_x, R, present), h._ptrs(h.recv_scales_phys, R, present) if use_fp8 else None,
                              count_ptrs, h._factor.data_ptr(), h._ptrs(h.expert_out, R), H, 0, T, E, h._stream(None))
        torch.cuda.synchronize()
        got = h.expert_out.cpu()
        for r in range(R):
            if r == absent:
                assert bool((got[r].view(torch.int16) == FILL).all()), f"rank {r} takes no part but was written"
            else:
                assert torch.equal(got[r].view(torch.int16), want[r].view(torch.int16)), f"rank {r}"


@pytest.mark.parametrize("experts", [4096, 4098])
def test_more_experts_than_a_block_looks_through(gpu_device, experts):
    cfg = EPConfig("experts", 2, 1, 128, experts, 1, False)
    announce(f"cast back with {experts} experts")
    h = WorldHarness(cfg)
    h.alloc_dispatch_outputs(poison=False)
    h.alloc_combine_io()
    h.recv_count.zero_()
    if experts <= 4096:
        h.cast_back(None)
    else:
        with pytest.raises(RuntimeError):
            h.cast_back(None)
    torch.cuda.synchronize()
