"""The channel matrices of a V1 handle, counted in the layout launch, at the edges of the count: fewer tokens than channels, one
channel, more channels than a wavefront has lanes, channels longer than a trip of 512 tokens, one chunk and several."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle
from test_gpu_intranode import _check_handle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_topk", [True, False], ids=["topk", "mask"])
@pytest.mark.parametrize("T,R,num_sms", [(1, 8, 24), (3, 2, 2), (255, 8, 256), (257, 5, 130), (1025, 8, 2), (5000, 8, 8)])
def test_channel_matrices(T, R, num_sms, with_topk):
    import deep_ep
    E, K = 8 * R, 4
    case = rc.small("channels", T, 128, E, R, K, seed=T, masked_ratio=0.3)
    rank = R // 2
    buf = deep_ep.Buffer(deep_ep.LogicalGroup(rank, R))
    idx = case.topk_idx.cuda()
    per_rank, _, per_expert, mask, _ = buf.get_dispatch_layout(idx, E)
    ref = oracle.intranode_dispatch(case.x, oracle.layout(case.topk_idx, E, R)[2], case.topk_idx if with_topk else None,
                                    case.topk_weights if with_topk else None, E, R, rank, 1, num_sms // 2)
    kw = dict(topk_idx=idx, topk_weights=case.topk_weights.cuda()) if with_topk else {}
    for _ in range(2):
        recv, _, _, _, handle, _ = buf.dispatch(case.x.cuda(), num_tokens_per_rank=per_rank, is_token_in_rank=mask,
                                                num_tokens_per_expert=per_expert, config=deep_ep.Config(num_sms, 6, 256), **kw)
        _check_handle(handle, ref, num_sms // 2)
        assert torch.equal(recv.cpu().view(torch.int16), ref.recv_x.view(torch.int16))
