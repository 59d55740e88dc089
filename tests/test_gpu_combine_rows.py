"""The combine at the edges of its row reads and of its routing loads: hidden sizes that end inside, at and past a column tile,
one to 65 ranks (a wavefront's lanes hold the ends of 64 regions), one to 32 selections, tokens without any row."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle

pytestmark = pytest.mark.gpu

# T, H, E, R, K
SHAPES = {
    "one_vector": (5, 8, 4, 1, 1),
    "tile_minus_one_vector": (67, 504, 32, 4, 4),
    "whole_tile": (67, 512, 32, 2, 5),
    "tile_plus_one_vector": (67, 520, 48, 6, 9),
    "two_tiles_and_a_vector": (130, 1032, 128, 64, 8),
    "more_ranks_than_lanes": (130, 1024, 130, 65, 12),
    "many_selections": (33, 1544, 96, 32, 32),
}


@pytest.mark.parametrize("expand", [False, True])
@pytest.mark.parametrize("reduce_in_rank", [True, False])
@pytest.mark.parametrize("name", SHAPES)
def test_combine_reads_its_rows(name, reduce_in_rank, expand):
    import deep_ep
    T, H, E, R, K = SHAPES[name]
    case = rc.small(name, T, H, E, R, K, seed=60, masked_ratio=0.3)
    case.topk_idx[T // 2] = -1                                             # a token that goes nowhere
    case.topk_weights[T // 2] = 0
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K,
                                allow_multiple_reduction=reduce_in_rank)
    recv_x, _, recv_w, handle, _ = buf.dispatch(case.x.cuda(), case.topk_idx.cuda(), case.topk_weights.cuda(), num_experts=E,
                                                do_expand=expand)
    gen = torch.Generator().manual_seed(61)
    y = torch.randn(recv_x.shape, generator=gen).to(torch.bfloat16)
    biases = tuple(torch.randn((T, H), generator=gen).to(torch.bfloat16) for _ in range(2))
    out, out_w, _ = buf.combine(y.cuda(), handle, topk_weights=recv_w, bias=tuple(b.cuda() for b in biases))
    ref, ref_w = oracle.combine(y, case.topk_idx, handle.recv_src_metadata.cpu(), handle.dst_buffer_slot_idx.cpu(),
                                handle.psum_num_recv_tokens_per_scaleup_rank.cpu(), E, R, 0, T, topk_weights=recv_w.cpu(), bias=biases,
                                do_expand=expand, allow_multiple_reduction=reduce_in_rank)
    # the order of the sums is fixed and there is one rounding: equal up to the sign of a zero
    assert torch.equal((out.cpu() + 0.0).view(torch.int16), (ref + 0.0).view(torch.int16))
    assert torch.equal(out_w.cpu(), ref_w)
    buf.check_device_status()


def test_a_handle_is_what_has_its_fields():
    """A combine takes whatever carries the reference's handle fields, also without the one this package adds."""
    import types

    import deep_ep
    c = rc.small("fields", 40, 128, 16, 4, 3, seed=3)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, c.R), num_max_tokens_per_rank=40, hidden=128, num_topk=3)
    recv, _, w, handle, _ = buf.dispatch(c.x.cuda(), c.topk_idx.cuda(), c.topk_weights.cuda(), num_experts=c.E)
    like = types.SimpleNamespace(**{k: v for k, v in vars(handle).items() if k != "rows_copied"})
    for a, b in zip(buf.combine(recv, handle, topk_weights=w)[:2], buf.combine(recv, like, topk_weights=w)[:2]):
        assert torch.equal(a, b)
