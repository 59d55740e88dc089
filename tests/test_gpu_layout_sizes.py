"""The layout pass at the sizes where it changes its way of working: one chunk of 256 tokens (handed over in LDS) and more, 16 and
32 chunks (columns held in registers), 48 and one more (sixteen a trip beyond), 64 ranks (membership by ballot), 8 and 12 routing
lanes (kernel variants), more experts than threads (the general publishing step).  Counts, prefix sums and placements are
integers: exactly the oracle's."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle

pytestmark = pytest.mark.gpu

SHAPES = [  # T, K, E, R
    (1, 8, 256, 8), (256, 8, 256, 8), (257, 8, 256, 8), (255, 12, 256, 64), (256, 3, 65, 65), (256, 8, 320, 8), (100, 1, 1, 1),
    (4096, 8, 256, 16), (4097, 9, 256, 17), (1237, 13, 72, 6), (8193, 8, 256, 32), (8192, 8, 320, 64), (16385, 8, 128, 64),
    (2048, 2, 130, 65), (12288, 4, 64, 8), (12289, 4, 64, 8),
]


@pytest.mark.parametrize("expand", [False, True], ids=["compact", "expanded"])
@pytest.mark.parametrize("T,K,E,R", [s if s[2] % s[3] == 0 else (s[0], s[1], s[2] // s[3] * s[3], s[3]) for s in SHAPES])
def test_layout(T, K, E, R, expand):
    import deep_ep
    case = rc.small("layout", T, 16, E, R, K, seed=T + K, masked_ratio=0.1)
    alignment = 8 if expand else 1
    ref = oracle.dispatch(case.x, case.topk_idx, case.topk_weights, E, R, 0, T, do_expand=expand, expert_alignment=alignment)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=16, num_topk=K)
    idx, w = case.topk_idx.cuda(), case.topk_weights.cuda()
    for _ in range(2):
        _, recv_idx, _, handle, _ = buf.dispatch(case.x.cuda(), idx, w, num_experts=E, do_expand=expand, expert_alignment=alignment)
        assert handle.num_recv_tokens == ref.num_recv_tokens
        assert torch.equal(handle.psum_num_recv_tokens_per_scaleup_rank.cpu(), ref.psum_num_recv_tokens_per_scaleup_rank)
        assert torch.equal(handle.psum_num_recv_tokens_per_expert.cpu(), ref.psum_num_recv_tokens_per_expert)
        assert torch.equal(handle.num_unaligned_recv_tokens_per_expert.cpu(), ref.num_unaligned_recv_tokens_per_expert)
        assert torch.equal(handle.dst_buffer_slot_idx.cpu(), ref.dst_buffer_slot_idx)
        assert torch.equal(handle.recv_src_metadata.cpu(), ref.recv_src_metadata)
