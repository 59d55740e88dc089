"""A call that throws when its layout is already queued - here: rows of no channels, which only the move launch refuses - leaves the
buffer fit for the next call, however late that layout runs."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle

pytestmark = pytest.mark.gpu
E, R, K, H = 64, 8, 6, 256


def _buffer(surface):
    import deep_ep
    group = deep_ep.LogicalGroup(0, R)
    return deep_ep.Buffer(group) if surface == "legacy" else deep_ep.ElasticBuffer(group, num_max_tokens_per_rank=1024, hidden=H, num_topk=K)


def _dispatch(buf, x, idx, w, **kw):
    import deep_ep
    if isinstance(buf, deep_ep.Buffer):
        if "layout" not in kw:
            kw["layout"] = buf.get_dispatch_layout(idx, E)
        per_rank, _, per_expert, mask, _ = kw.pop("layout")
        return buf.dispatch(x, num_tokens_per_rank=per_rank, is_token_in_rank=mask, num_tokens_per_expert=per_expert, topk_idx=idx,
                            topk_weights=w, **kw)
    kw.pop("layout", None)
    return buf.dispatch(x, idx, w, num_experts=E, **kw)


def _throw_behind_a_busy_stream(buf, surface):
    """A call on the communication stream, behind tens of milliseconds of products on another stream, that throws with its layout
    queued.  Returns the event behind the products and the inputs."""
    case = rc.small("thrown", 1024, 16, E, R, K, seed=70)
    idx, w = case.topk_idx.cuda(), case.topk_weights.cuda()
    layout = buf.get_dispatch_layout(idx, E)
    overlap = {"async_finish": True} if surface == "legacy" else {"async_with_compute_stream": True}
    x = torch.empty((1024, 0), dtype=torch.bfloat16, device="cuda")
    a, b = torch.randn((8192, 8192), device="cuda"), torch.empty((8192, 8192), device="cuda")
    busy = torch.cuda.Stream()
    for products in (1, 12):                      # the first pass makes what is allocated once: allocations may wait for the GPU
        _dispatch(buf, case.x.cuda(), idx, w, layout=layout)
        torch.cuda.synchronize()
        with torch.cuda.stream(busy):
            for _ in range(products):
                torch.mm(a, a, out=b)
            until = buf.capture()
            end = torch.cuda.Event()
            end.record()
        with pytest.raises(RuntimeError, match="hidden|multiple of 16"):
            _dispatch(buf, x, idx, w, layout=layout, previous_event=until, allocate_on_comm_stream=True, **overlap)
    assert not end.query(), "the products were over too early for this test to say anything"
    return end, (idx, w, layout, a, b)


@pytest.mark.parametrize("surface", ["elastic", "legacy"])
def test_counts_of_a_thrown_call_are_not_taken_for_the_next_ones(surface):
    buf = _buffer(surface)
    case = rc.small("next", 40, H, E, R, K, seed=71, masked_ratio=0.2)
    x, idx, w = case.x.cuda(), case.topk_idx.cuda(), case.topk_weights.cuda()
    ref = oracle.dispatch(case.x, case.topk_idx, case.topk_weights, E, R, 0, 1024)
    keep = _throw_behind_a_busy_stream(buf, surface)
    recv_x, recv_idx, _, *rest = _dispatch(buf, x, idx, w)
    per_expert = rest[0] if surface == "legacy" else rest[0].num_recv_tokens_per_expert_list
    assert tuple(recv_x.shape) == (ref.num_recv_tokens, H)
    assert list(per_expert) == ref.num_unaligned_recv_tokens_per_expert.tolist()
    assert torch.equal(recv_x.cpu().view(torch.int16), ref.recv_x.view(torch.int16))
    assert torch.equal(recv_idx.cpu(), ref.recv_topk_idx)
    del keep


@pytest.mark.parametrize("surface", ["elastic", "legacy"])
def test_work_after_a_thrown_call_is_ordered_behind_it(surface):
    """The thrown call's launches read its inputs and use the buffer's workspace: neither what follows on the caller's stream nor the
    next call on the buffer, on whatever stream, may run before them."""
    buf = _buffer(surface)
    end, keep = _throw_behind_a_busy_stream(buf, surface)
    after = torch.cuda.Event()
    after.record()
    after.synchronize()
    assert end.query(), "the caller's stream did not wait for the launches of the call that threw"

    end, keep = _throw_behind_a_busy_stream(buf, surface)
    other = torch.cuda.Stream()
    with torch.cuda.stream(other):
        buf.get_dispatch_layout(keep[0], E)
        after.record()
    after.synchronize()
    assert end.query(), "the next call on the buffer did not wait for the launches of the call that threw"


def test_a_low_latency_call_does_not_stand_for_the_dispatches_before_it():
    """It uses a workspace of its own: a later call on its stream still waits for dispatches queued on another."""
    import deep_ep
    buf = deep_ep.Buffer(deep_ep.LogicalGroup(0, R), low_latency_mode=True)
    case = rc.small("behind", 64, 512, E, R, K, seed=72)
    x, idx, w = case.x.cuda(), case.topk_idx.cuda(), case.topk_weights.cuda()
    a, b = torch.randn((8192, 8192), device="cuda"), torch.empty((8192, 8192), device="cuda")
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    for products in (1, 12):
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            for _ in range(products):
                torch.mm(a, a, out=b)
            buf.get_dispatch_layout(idx, E)
            end = torch.cuda.Event()
            end.record()
        with torch.cuda.stream(second):
            buf.low_latency_dispatch(x, idx, 64, E, use_fp8=False)
            assert products == 1 or not end.query(), "the products were over too early for this test to say anything"
            buf.get_dispatch_layout(idx, E)
            after = torch.cuda.Event()
            after.record()
        after.synchronize()
        assert end.query()
