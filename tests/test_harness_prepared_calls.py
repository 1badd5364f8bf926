"""The whole-world driver keeps marshalled calls: one made from tensors that have been replaced since, or from other
token counts, is not used again, and only so many are kept.  (No GPU: a world that writes down what it is given.)"""
from types import SimpleNamespace

import pytest
import torch

from mooncake_amd.harness import WorldHarness
from mooncake_amd.workloads import EPConfig

STREAM = SimpleNamespace(cuda_stream=0)


class World:
    num_ranks = 2

    def __init__(self):
        self.prepared, self.called = 0, []

    def _prepare(self, *args):
        self.prepared += 1
        return lambda stream, phases: self.called.append(args)

    prepare_dispatch = prepare_combine = prepare_combine_packed = _prepare


def harness(world):
    cfg = EPConfig("keys", 2, 6, 128, 4, 2, True)
    h = WorldHarness(cfg, device="cpu", world=world)
    h.load({"x": torch.zeros(2, 6, 128, dtype=torch.bfloat16), "topk_idx": torch.zeros(2, 6, 2, dtype=torch.int64),
            "topk_weights": torch.zeros(2, 6, 2)})
    h.alloc_dispatch_outputs()
    h.alloc_combine_io()
    return h


CALLS = {
    "dispatch": (lambda h: h.dispatch(stream=STREAM),
                 ("x", "topk_idx", "recv_x", "recv_scales_phys", "recv_count", "src_info", "layout_range")),
    "combine": (lambda h: h.combine(stream=STREAM),
                ("expert_out", "topk_idx", "topk_weights", "src_info", "layout_range", "active_ranks", "combined")),
    "combine_packed": (lambda h: h.combine_packed(stream=STREAM),
                       ("recv_x", "recv_scales_phys", "topk_idx", "topk_weights", "src_info", "layout_range",
                        "active_ranks", "combined")),
}


@pytest.mark.parametrize("kind", CALLS)
def test_a_call_is_made_of_the_tensors_it_has_now(kind):
    call, fields = CALLS[kind]
    world = World()
    h = harness(world)
    call(h)
    call(h)
    assert world.prepared == 1
    kept = []
    for name in fields:
        old = getattr(h, name)
        kept.append(old)                                   # (so that the new one has an address of its own)
        setattr(h, name, torch.empty_like(old))
        call(h)
        assert any(getattr(h, name)[1].data_ptr() in a for a in world.called[-1] if isinstance(a, list)), name
    h.num_tokens[1] = 3
    call(h)
    assert any(a == [6, 3] for a in world.called[-1] if isinstance(a, list))
    assert world.prepared == 2 + len(fields)


def test_ranks_spaced_otherwise_from_the_same_address():
    world = World()
    h = harness(world)
    wide = torch.zeros(2, 2, 6, 2, dtype=torch.int64)
    h.topk_idx = wide[0]
    h.dispatch(stream=STREAM)
    h.topk_idx = wide[:, 0]
    h.dispatch(stream=STREAM)
    assert world.called[-1][1] == [wide[0, 0].data_ptr(), wide[1, 0].data_ptr()]


def test_only_so_many_are_kept():
    world = World()
    h = harness(world)
    xs = [torch.zeros_like(h.x) for _ in range(h._MOST_PREPARED + 10)]
    for x in xs:
        h.x = x
        h.dispatch(stream=STREAM)
    assert len(h._prepared) == h._MOST_PREPARED
    h.dispatch(stream=STREAM)
    assert world.prepared == len(xs)                       # the latest is among them
