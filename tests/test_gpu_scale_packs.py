"""Scale packs of FP8 rows moved as they are: 64 and more to a row (a wavefront's lanes hold the first 64), their strides, and rows
of one KB in a call so large that a wavefront stores them row by row.  Every row and pack is its token's."""
import pytest
import torch

import routing_cases as rc

pytestmark = pytest.mark.gpu

# T, H, R, K
SHAPES = {"a_wavefront": (130, 8192, 8, 4), "one_beyond": (67, 8320, 4, 3), "many_beyond": (33, 20480, 8, 4), "row_by_row": (16411, 1024, 8, 8)}


@pytest.mark.parametrize("mode", ["exact", "one_launch", "expanded", "column_major_input", "legacy"])
@pytest.mark.parametrize("shape", SHAPES)
def test_packs_are_the_tokens(shape, mode):
    import deep_ep
    from deep_ep.utils.math import per_token_cast_to_fp8
    T, H, R, K = SHAPES[shape]
    E = 64
    case = rc.small(shape, T, 16, E, R, K, seed=80, masked_ratio=0.1)
    idx, w = case.topk_idx.cuda(), case.topk_weights.cuda()
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(81), device="cuda", dtype=torch.bfloat16)
    q, sf = per_token_cast_to_fp8(x)
    given = sf.T.contiguous().T if mode == "column_major_input" else sf
    if mode == "legacy":
        buf = deep_ep.Buffer(deep_ep.LogicalGroup(0, R))
        per_rank, _, per_expert, mask, _ = buf.get_dispatch_layout(idx, E)
        (recv, recv_sf), _, _, _, handle, _ = buf.dispatch((q, given), num_tokens_per_rank=per_rank, is_token_in_rank=mask,
                                                           num_tokens_per_expert=per_expert, topk_idx=idx, topk_weights=w)
        rows, tokens = torch.arange(recv.shape[0], device="cuda"), handle[3].long()
    else:
        buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
        (recv, recv_sf), _, _, handle, _ = buf.dispatch((q, given), idx, w, num_experts=E, do_expand=mode == "expanded",
                                                        do_cpu_sync=mode != "one_launch")
        meta = handle.recv_src_metadata[:int(handle.psum_num_recv_tokens_per_scaleup_rank[-1])]
        if mode == "expanded":
            at = meta[:, 2:]
            rows, tokens = at[at >= 0].long(), meta[:, :1].expand_as(at)[at >= 0].long()
        else:
            rows, tokens = torch.arange(meta.shape[0], device="cuda"), meta[:, 0].long()
    routed = (idx >= 0).sum() if mode == "expanded" else sum(int((idx // (E // R) == r).any(1).sum()) for r in range(R))
    assert rows.numel() == int(routed)
    assert torch.equal(recv.view(torch.uint8)[rows], q.view(torch.uint8)[tokens])
    assert torch.equal(recv_sf[rows], sf[tokens])
    if mode != "legacy":
        buf.check_device_status()
