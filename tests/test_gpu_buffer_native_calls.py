"""The Python `Buffer`'s dispatch and combine through the compiled module: the outputs have the shapes, strides and
types of the Python statement of the same call, a set of outputs is offered again only when nothing refers to any of
its storages, and what the Python statement refuses is refused with the same exception."""
import gc

import pytest
import torch

from mooncake_amd import Buffer, LogicalGroup
from tests.gpu_util import announce

pytestmark = pytest.mark.gpu

T, H, E, K = 12, 256, 8, 3


def buffers(native, ranks=1):
    _, groups = LogicalGroup.make_world(ranks)
    size = Buffer.get_ep_buffer_size_hint(2 * T, H, ranks, E)
    bufs = [Buffer(g, size) for g in groups]
    for b in bufs:
        assert b._dispatch_tensors is not None and b._combine_tensors is not None
        if not native:
            b._dispatch_tensors = b._combine_tensors = None
    return bufs


def inputs(seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).cuda()
    idx = torch.randn(T, E, generator=g).topk(K)[1].cuda()
    return x, idx, torch.rand(T, K, generator=g).cuda()


def described(t):
    return t.shape, t.stride(), t.dtype, t.device


@pytest.mark.parametrize("fp8", [True, False], ids=["fp8", "bf16"])
@pytest.mark.parametrize("mode", ["default", "async", "hook"])
def test_both_statements_of_a_call_agree(gpu_device, fp8, mode):
    announce(f"Buffer calls, native against Python: fp8={fp8} {mode}")
    kw = {"async_finish": mode == "async", "return_recv_hook": mode == "hook"}
    results = []
    for native in (True, False):
        buf = buffers(native)[0]
        x, idx, w = inputs()
        recv, count, handle, event, hook = buf.dispatch(x, idx, None, T, E, -1, use_fp8=fp8, **kw)
        if hook is not None:
            hook()
        rows = torch.ones((E, T, H), dtype=torch.bfloat16, device=gpu_device)
        out, event2, hook2 = buf.combine(rows, idx, w, torch.ones(1, dtype=torch.int32, device=gpu_device), -1, handle, **kw)
        if hook2 is not None:
            hook2()
        torch.cuda.synchronize()
        assert (event.event is not None) == (event2.event is not None) == (mode == "async")
        results.append((recv if fp8 else (recv,), count, handle, out))
    (ra, ca, ha, oa), (rb, cb, hb, ob) = results
    for a, b in zip((*ra, ca, ha[0], ha[1], oa), (*rb, cb, hb[0], hb[1], ob)):
        assert described(a) == described(b)
    assert ha[2:] == hb[2:] and torch.equal(ca, cb) and torch.equal(ha[1], hb[1]) and torch.equal(oa, ob)
    for e, n in enumerate(ca.tolist()):
        assert torch.equal(ha[0][e, :n], hb[0][e, :n])
        for a, b in zip(ra, rb):
            a, b = (t[e, :n].contiguous().view(torch.uint8) for t in (a, b))
            assert torch.equal(a, b)


def test_outputs_are_offered_again_only_when_nothing_refers_to_them(gpu_device):
    announce("Buffer outputs: recycling")
    buf = buffers(True)[0]
    x, idx, _ = inputs()

    def call():
        return buf.dispatch(x, idx, None, T, E, -1, use_fp8=True)[:3]

    a = call()
    first = a[0][0].data_ptr()
    b = call()                                              # a is held
    assert b[0][0].data_ptr() != first
    view = a[0][1][0].view(torch.int32)                     # a view of the scales keeps the whole set
    del a
    gc.collect()
    assert call()[0][0].data_ptr() != first
    del view
    gc.collect()
    c = call()
    assert c[0][0].data_ptr() == first
    c[2][0].untyped_storage().resize_(0)                    # and a storage of another size is not offered
    del c
    gc.collect()
    d = call()
    assert d[0][0].data_ptr() != first and d[2][0].untyped_storage().nbytes() == E * T * 4


@pytest.mark.parametrize("native", [True, False], ids=["native", "python"])
def test_refusals(gpu_device, native):
    announce(f"Buffer refusals, native={native}")
    buf = buffers(native)[0]
    x, idx, w = inputs()
    bad = [(x.float(), idx, None), (x, idx.int(), None), (x[:, :128], idx, None), (x[:5], idx, None), (x[0], idx, None),
           (x, idx.t().contiguous().t(), None), (x, idx, torch.ones(1, device=gpu_device)),
           (x[:, :64].contiguous(), idx, None)]
    for args in bad:
        with pytest.raises(AssertionError):
            buf.dispatch(*args, T, E, -1, use_fp8=True)
    with pytest.raises(AssertionError):
        buf.dispatch(x, idx, None, T - 1, E, -1)
    if native:                                              # (the Python statement allocates its outputs first)
        with pytest.raises(TypeError):
            buf.dispatch(x[:4], idx[:4], None, 2 ** 32, E, -1)
    _, _, handle, _, _ = buf.dispatch(x, idx, None, T, E, -1, use_fp8=True)
    rows = torch.zeros((E, T, H), dtype=torch.bfloat16, device=gpu_device)
    out = torch.empty((T, H), dtype=torch.bfloat16, device=gpu_device)
    good = dict(x=rows, topk_idx=idx, topk_weights=w, active_ranks=None, timeout_us=-1, handle=handle, out=out)
    for name, value in (("x", rows[:, :4]), ("x", rows.float()), ("topk_idx", idx[:4]), ("topk_weights", w.double()),
                        ("handle", (handle[0][:4], *handle[1:])), ("handle", (handle[0], handle[1].int(), *handle[2:])),
                        ("handle", (*handle[:3], 128, E)), ("out", out[:4]), ("out", out.float())):
        with pytest.raises(AssertionError):
            buf.combine(**dict(good, **{name: value}))
    # an active_ranks tensor of another size stands for everybody alive
    got = buf.combine(**dict(good, active_ranks=torch.zeros(3, dtype=torch.int32, device=gpu_device)))[0]
    assert got.data_ptr() == out.data_ptr()
    torch.cuda.synchronize()
