"""Whole-world calls straight from stacked tensors (the compiled module reads every rank's address off them) against the
calls marshalled in Python: the same results for full, ragged and partly silent worlds, ranks at any spacing, tensor
subclasses, an fp8 and a bf16 payload, with and without a factor; and the same refusals."""
import pytest
import torch

from mooncake_amd.harness import WorldHarness
from mooncake_amd.workloads import EPConfig, generate
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu

R, T = 4, 12


class Own(torch.Tensor):
    pass


def cycle(h, present, factor):
    """Every whole-world call once; what they wrote."""
    out = []
    h.dispatch(present=present)
    out += [h.recv_count, h.src_info, h.layout_range, h.recv_x] + ([h.recv_scales_phys] if h.cfg.use_fp8 else [])
    h.cast_back(factor, present=present)
    out.append(h.expert_out)
    for call in (lambda: h.combine(present=present), lambda: h.combine_packed(factor, present=present)):
        h.combined.fill_(7.0)
        call()
        out.append(h.combined.clone())
    torch.cuda.synchronize()
    return [t.cpu().contiguous().view(torch.uint8) for t in out]


def harness(cfg, data, nt, spaced):
    h = WorldHarness(cfg, num_tokens=nt)
    h.load(data)
    if spaced:                                      # ranks further apart than a rank's tensor is long
        for name in ("x", "topk_idx", "topk_weights"):
            t = getattr(h, name)
            wide = t.new_zeros((R, 3) + tuple(t.shape[1:]))
            wide[:, 1] = t
            setattr(h, name, wide[:, 1])
    h.alloc_dispatch_outputs(poison=True)
    h.alloc_combine_io()
    h.expert_out.zero_()
    return h


@pytest.mark.parametrize("use_fp8", [True, False], ids=["fp8", "bf16"])
@pytest.mark.parametrize("how", ["full", "ragged", "silent", "spaced", "subclass"])
def test_stacked_calls_do_what_marshalled_ones_do(gpu_device, monkeypatch, use_fp8, how):
    announce(f"stacked calls {how} fp8={use_fp8}")
    cfg = EPConfig("stacked", R, T, 640, 8, 3, use_fp8)
    data = generate(cfg, seed=5)
    nt = [T, 0, 5, 11] if how == "ragged" else None
    present = [1, 0, True, 1] if how == "silent" else None
    got = []
    for stacked in (True, False):
        h = harness(cfg, data, nt, how == "spaced")
        if how == "subclass":
            h.x = h.x.as_subclass(Own)
        if not stacked:
            monkeypatch.setattr(h, "_stacked", lambda ranks: None)
        factor = torch.arange(8).float() * 0.25 + 0.5
        got.append(cycle(h, present, factor) + cycle(h, present, None))
        assert (len(h._prepared) > 0) == (not stacked or how == "subclass")      # (marshalled calls are kept)
    assert all(torch.equal(a, b) for a, b in zip(*got))


def test_stacked_calls_refuse_what_marshalled_ones_refuse(gpu_device, monkeypatch):
    cfg = EPConfig("refused", R, T, 640, 8, 3, False)
    data = generate(cfg, seed=6)
    for stacked in (True, False):
        announce(f"stacked calls: refusals, stacked={stacked}")
        h = harness(cfg, data, None, False)
        if not stacked:
            monkeypatch.setattr(h, "_stacked", lambda ranks: None)
        x, tokens = h.x, h.num_tokens
        h.x = x[:R - 1]
        with pytest.raises(IndexError):
            h.dispatch()
        h.x, h.num_tokens = x, tokens[:R - 1]
        with pytest.raises(ValueError):
            h.dispatch()
        h.num_tokens = [T + 1] + tokens[1:]
        with pytest.raises(RuntimeError):
            h.combine()
        h.num_tokens, h.topk_idx = tokens, None
        with pytest.raises(RuntimeError):
            h.dispatch()


def test_forms_that_marshalled_calls_take(gpu_device, monkeypatch):
    """Ranks that take part and token counts in other forms than lists of numbers, and tensors that end with the last
    rank that takes part."""
    import numpy as np

    cfg = EPConfig("forms", R, T, 640, 8, 3, True)
    data = generate(cfg, seed=7)
    on, nt = [1, 1, 1, 0], [T, 0, 5, 11]
    forms = {
        "lists": (on, nt),
        "tensors": (torch.tensor(on), torch.tensor(nt)),
        "on_the_gpu": (torch.tensor(on, device=gpu_device), list(torch.tensor(nt, device=gpu_device))),
        "arrays": (np.array(on), np.array(nt, dtype=np.int64)),
        "tuples": (tuple(map(bool, on)), tuple(nt)),
        "by_rank": (dict(enumerate(on)), [float(n) for n in nt]),
        "texts": (["yes", "yes", "yes", ""], [np.int32(n) for n in nt]),
        "longer": (on + [1], nt),
    }
    got = {}
    for stacked in (True, False):
        for name, (present, tokens) in forms.items():
            announce(f"stacked calls: {name}, stacked={stacked}")
            h = harness(cfg, data, nt, False)
            h.num_tokens = tokens
            if not stacked:
                monkeypatch.setattr(h, "_stacked", lambda ranks: None)
            got[name, stacked] = cycle(h, present, None)
        announce(f"stacked calls: tensors of three ranks, stacked={stacked}")
        h = harness(cfg, data, nt, False)
        if not stacked:
            monkeypatch.setattr(h, "_stacked", lambda ranks: None)
        for name in ("recv_x", "recv_scales_phys"):
            setattr(h, name, getattr(h, name)[:R - 1])
        h.expert_out.zero_()
        h.dispatch(present=on)
        h.cast_back(present=on)
        h.combine(present=on)
        h.combine_packed(present=on)
        torch.cuda.synchronize()
        got["three", stacked] = [h.expert_out.cpu().contiguous().view(torch.uint8)]
    for name in forms:
        for stacked in (True, False):
            assert all(torch.equal(a, b) for a, b in zip(got[name, stacked], got["lists", False])), (name, stacked)
    assert torch.equal(got["three", True][0], got["three", False][0])
