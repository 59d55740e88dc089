"""The layout launch with every kernel for a number of selections, in one workgroup of one and of two chunks and in several, on both sides of
the ranks it takes by ballot (16) and by sets of 32 and 64 bits; every word it leaves against the oracle, the callers' indices copied as they are,
misaligned too, and bad routing flagged wherever it stands."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle
from test_gpu_parity import assert_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 13, 17, 21, 32])
@pytest.mark.parametrize("T,R,E_l", [(255, 16, 4), (257, 17, 4), (512, 8, 39), (511, 8, 40), (513, 32, 3), (300, 64, 2), (261, 65, 2)])
def test_layout_of_every_kernel(T, R, E_l, K):
    import deep_ep
    E = R * E_l
    case = rc.small("topk", T, 16, E, R, K, seed=T + K, masked_ratio=0.1)
    case.topk_idx[case.topk_idx == 5] = -(1 << 40)            # negative, however large: no expert
    case.topk_weights[case.topk_idx < 0] = 0.0
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=16, num_topk=K)
    x, w = case.x.cuda(), case.topk_weights.cuda()
    odd = torch.empty(T * K + 1, dtype=torch.int64, device="cuda")
    odd[1:] = case.topk_idx.cuda().flatten()
    for idx in (case.topk_idx.cuda(), odd[1:].view(T, K)):    # on 16 bytes, and 8 past them
        for expand in (False, True):
            ref = oracle.dispatch(case.x, case.topk_idx, case.topk_weights, E, R, 0, T, do_expand=expand, expert_alignment=3 if expand else 1)
            recv, _, _, handle, _ = buf.dispatch(x, idx, w, num_experts=E, do_expand=expand, expert_alignment=3 if expand else 1)
            assert_equal(handle.dst_buffer_slot_idx, ref.dst_buffer_slot_idx, "dst_buffer_slot_idx")
            assert_equal(handle.psum_num_recv_tokens_per_expert, ref.psum_num_recv_tokens_per_expert, "psum per expert")
            assert_equal(handle.psum_num_recv_tokens_per_scaleup_rank, ref.psum_num_recv_tokens_per_scaleup_rank, "psum per rank")
            assert_equal(handle.recv_src_metadata, ref.recv_src_metadata, "recv_src_metadata")
            assert torch.equal(handle.topk_idx, idx)
        counts = buf.get_dispatch_layout(idx, E)
        of = oracle.layout(case.topk_idx, E, R)
        assert_equal(counts[0], of[0], "num_tokens_per_rank")
        assert_equal(counts[2], of[1], "num_tokens_per_expert")
        assert_equal(counts[3], of[2], "is_token_in_rank")
    buf.check_device_status()


@pytest.mark.parametrize("K", [1, 3, 8, 9])
@pytest.mark.parametrize("T", [200, 300, 700])
def test_bad_routing_is_flagged(T, K):
    import deep_ep
    E, R = 48, 4
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=16, num_topk=K)
    good = torch.rand((T, E), device="cuda").topk(K, dim=1).indices
    x, w = torch.zeros((T, 16), dtype=torch.bfloat16, device="cuda"), torch.rand((T, K), device="cuda")
    for token, lane in ((0, 0), (T - 1, K - 1)):
        for bad, says in ((E, "expert id"), ((1 << 32) + 3, "expert id"), (None, "twice")):
            if bad is None and K == 1:
                continue
            idx = good.clone()
            idx[token, lane] = idx[token, lane - 1] if bad is None else bad
            with pytest.raises(RuntimeError, match=says):
                buf.dispatch(x, idx, w, num_experts=E)
    buf.dispatch(x, good, w, num_experts=E)
    buf.check_device_status()
