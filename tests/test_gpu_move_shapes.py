"""Moves at the lines of their choice of a column tile, of the workgroups a CU holds and of rows stored in turn, one size or more for each outcome,
which is asked for: rows that end inside a vector group, a tile and on one, aligned and masked calls, every word against the token it came from."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle
from test_move_choice import combine, move, shape, v1_move

pytestmark = pytest.mark.gpu

CASES = {   # tokens, channels, experts, ranks, selections, payload, expanded, alignment: (tile, workgroups a CU holds or 0, rows stored in turn)
    "one_kb_by_wavefronts": ((1921, 4096, 64, 2, 2, "bf16", False, 1), (4, 0, 0)),               # 2 KB up to 1920 tokens: 30 wavefronts a CU
    "wide_by_wavefronts": ((1923, 4096, 64, 2, 2, "bf16", False, 1), (4, 0, 0)),
    "up_to_thirty_wavefronts": ((1919, 4096, 64, 2, 2, "bf16", False, 1), (2, 0, 0)),
    "up_to_four_wavefronts": ((341, 2888, 64, 8, 8, "bf16", False, 1), (1, 0, 0)),               # of 2 KB
    "past_four_wavefronts": ((342, 2888, 64, 8, 8, "bf16", False, 1), (2, 0, 0)),
    "whole_8kb_up_to_six_wavefronts": ((384, 4096, 64, 8, 8, "bf16", False, 1), (1, 0, 0)),
    "whole_8kb_past_six_wavefronts": ((385, 4096, 64, 8, 8, "bf16", False, 1), (2, 0, 0)),
    "eight_rows_up_to_15_wavefronts": ((548, 7168, 64, 8, 8, "bf16", True, 1), (1, 0, 0)),
    "eight_rows_past_15_wavefronts": ((549, 7168, 64, 8, 8, "bf16", True, 1), (2, 0, 0)),
    "half_empty_two_kb": ((2362, 1064, 64, 8, 8, "bf16", False, 1), (1, 0, 0)),                  # rows of 2.1 KB
    "two_kb_by_wavefronts": ((3847, 2040, 64, 8, 6, "bf16", False, 1), (2, 0, 0)),
    "ragged_two_workgroups": ((2237, 5112, 64, 8, 8, "bf16", False, 1), (2, 2, 0)),              # 120 MB of rows, out of the cache
    "ragged_three_workgroups": ((3301, 5112, 64, 4, 4, "bf16", False, 1), (4, 0, 0)),            # 92 MB, in it: the widest tile
    "ragged_three_rows": ((4507, 5112, 64, 4, 4, "bf16", False, 1), (2, 3, 0)),                  # 126 MB, 2.7 rows a token
    "ragged_large_input": ((9001, 5112, 64, 8, 6, "bf16", False, 1), (2, 3, 0)),                 # 92 MB of input, 4.4 rows
    "ragged_three_kb": ((10007, 1048, 256, 32, 8, "bf16", False, 1), (4, 2, 0)),                 # the last vectors of a row absent
    "ragged_four_kb": ((8009, 2040, 64, 8, 8, "bf16", False, 1), (4, 2, 0)),
    "ragged_two_rows": ((9001, 3976, 64, 8, 2, "bf16", False, 1), (2, 5, 0)),
    "ragged_two_rows_many_ranks": ((9001, 3976, 64, 64, 2, "bf16", False, 1), (2, 4, 0)),
    "ragged_one_row": ((9001, 8008, 64, 8, 1, "bf16", False, 1), (2, 0, 0)),
    "expanded_one_kb": ((7507, 2552, 64, 8, 8, "bf16", True, 1), (2, 2, 0)),                     # eight rows: 2 KB
    "expanded_nine_rows": ((4927, 5080, 72, 8, 9, "bf16", True, 1), (1, 2, 0)),                  # 451 MB
    "expanded_two_kb": ((4001, 2552, 64, 8, 8, "bf16", True, 16), (2, 2, 0)),
    "whole_five_workgroups": ((6607, 2048, 64, 8, 8, "bf16", False, 1), (1, 5, 0)),
    "whole_four_workgroups": ((6607, 2048, 256, 32, 8, "bf16", False, 1), (1, 4, 0)),
    "whole_power_of_two": ((10007, 4096, 64, 8, 8, "bf16", False, 1), (1, 6, 1)),                # 430 MB of 8 KB, 5.3 rows
    "whole_power_of_two_four_rows": ((12503, 4096, 64, 8, 6, "bf16", False, 1), (2, 3, 0)),      # 4.4
    "whole_in_turn_no_limit": ((7507, 7168, 64, 8, 6, "bf16", False, 1), (1, 0, 1)),
    "whole_many_ranks": ((7001, 7168, 256, 64, 4, "bf16", False, 1), (2, 3, 0)),
    "fp8_whole_many_ranks": ((14003, 7168, 256, 64, 4, "fp8", False, 1), (2, 4, 0)),
    "whole_few_rows": ((9001, 4096, 64, 8, 4, "bf16", False, 1), (2, 4, 0)),
    "fp8_four_workgroups": ((20011, 3968, 64, 8, 6, "fp8", False, 1), (2, 4, 0)),
    "fp8_three_workgroups": ((17011, 3968, 64, 8, 8, "fp8", True, 1), (2, 3, 0)),
    "fp8_expanded_four_kb": ((6307, 3968, 64, 8, 8, "fp8", True, 1), (4, 0, 0)),                 # 200 MB
    "fp8_whole_in_turn": ((5003, 4096, 64, 8, 8, "fp8", False, 1), (1, 0, 1)),
    "fp8_whole_in_turn_six": ((3001, 5120, 256, 32, 8, "fp8", False, 1), (1, 6, 1)),
    "cast_five_workgroups": ((12007, 4992, 64, 8, 6, "cast", False, 1), (2, 5, 0)),
    "cast_four_workgroups": ((12007, 4992, 64, 8, 8, "cast", False, 1), (2, 4, 0)),
    "cast_four_of_one_kb": ((5003, 7168, 256, 32, 8, "cast", False, 1), (1, 4, 0)),
    "cast_three_workgroups": ((7001, 4992, 64, 8, 8, "cast", True, 1), (2, 3, 0)),
}


@pytest.mark.parametrize("name", CASES)
def test_every_word_is_its_tokens(name):
    import deep_ep
    from deep_ep.utils.math import per_token_cast_to_fp8
    (T, H, E, R, K, payload, expand, A), chosen = CASES[name]
    assert shape(move(payload, T, H, E, R, K, expanded=expand, alignment=A)) == chosen
    small = rc.small(name, T, 16, E, R, K, seed=60, masked_ratio=0.03)         # the routing, with a payload of 16 channels
    ref = oracle.dispatch(small.x, small.topk_idx, small.topk_weights, E, R, 0, T, do_expand=expand, expert_alignment=A)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(61), device="cuda", dtype=torch.bfloat16)
    pair = per_token_cast_to_fp8(x) if payload != "bf16" else (x,)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    recv, recv_idx, recv_w, handle, _ = buf.dispatch(pair if payload == "fp8" else x, small.topk_idx.cuda(), small.topk_weights.cuda(), num_experts=E,
                                                     do_expand=expand, expert_alignment=A, cast_to_fp8=payload == "cast")
    meta = handle.recv_src_metadata
    assert torch.equal(meta.cpu(), ref.recv_src_metadata)
    assert torch.equal(handle.dst_buffer_slot_idx.cpu(), ref.dst_buffer_slot_idx)
    if expand:
        rows = meta[:, 2:]
        at, tokens = rows[rows >= 0].long(), meta[:, :1].expand_as(rows)[rows >= 0].long()
        assert torch.equal(recv_w[at].cpu(), ref.recv_topk_weights[at.cpu()])
    else:
        tokens = meta[:, 0].long()
        at = torch.arange(tokens.numel(), device="cuda")
        assert torch.equal(recv_idx.cpu(), ref.recv_topk_idx) and torch.equal(recv_w.cpu(), ref.recv_topk_weights)
    for got, want in zip((recv,) if payload == "bf16" else recv, pair):
        assert torch.equal(got[at].view(torch.uint8), want[tokens].view(torch.uint8))
    buf.check_device_status()


@pytest.mark.parametrize("T,H,E,R,K,expand,tiles", [          # KB of the dispatch and of the combine
    (211, 7960, 64, 8, 8, False, (2, 2)), (1, 4096, 8, 4, 2, False, (2, 2)), (7, 2040, 64, 8, 8, False, (2, 2)),
    (352, 7168, 64, 8, 8, False, (2, 2)), (353, 7168, 64, 8, 8, False, (2, 2)),
    (804, 7168, 64, 8, 8, False, (2, 2)), (805, 7168, 64, 8, 8, False, (4, 2)),              # 22 wavefronts of 2 KB a CU
    (437, 7168, 256, 32, 8, False, (2, 2)), (439, 7168, 256, 32, 8, False, (2, 2)), (1409, 4096, 64, 8, 4, False, (4, 2)), (1407, 4088, 64, 8, 4, False, (2, 2)),
    (256, 4096, 64, 8, 8, False, (2, 2)), (257, 4096, 64, 8, 8, False, (1, 1)),              # four and six, rows of whole 8 KB
    (384, 4096, 64, 8, 8, False, (1, 1)), (385, 4096, 64, 8, 8, False, (2, 2)),
    (146, 7168, 64, 8, 8, True, (1, 1)), (147, 7168, 64, 8, 8, True, (2, 2)),                # eight rows a token: four
])
def test_rows_of_a_single_launch_and_their_sum(T, H, E, R, K, expand, tiles):
    import deep_ep
    s = move("bf16", T, H, E, R, K, expanded=expand, single=True)
    assert s.single_launch == 1 and (s.tile, combine(T, H, E, R, K, 2, expanded=expand)) == tiles
    small = rc.small("single", T, 16, E, R, K, seed=62, masked_ratio=0.05)
    ref = oracle.dispatch(small.x, small.topk_idx, small.topk_weights, E, R, 0, T, do_expand=expand)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(63), device="cuda", dtype=torch.bfloat16)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K, allow_multiple_reduction=not expand)
    recv, _, w, handle, _ = buf.dispatch(x, small.topk_idx.cuda(), small.topk_weights.cuda(), num_experts=E, do_expand=expand, do_cpu_sync=False)
    n = ref.recv_src_metadata.shape[0]
    meta = handle.recv_src_metadata[:n]
    assert torch.equal(meta.cpu(), ref.recv_src_metadata)
    rows = meta[:, 2:] if expand else torch.arange(n, device="cuda")[:, None]
    tokens = meta[:, :1].expand_as(rows)[rows >= 0].long()
    assert torch.equal(recv[rows[rows >= 0].long()].view(torch.int16), x[tokens].view(torch.int16))
    out, _, _ = buf.combine(recv, handle, topk_weights=w)
    count = torch.zeros(T, device="cuda").index_add_(0, tokens, torch.ones(tokens.numel(), device="cuda"))
    assert torch.equal(out, (x.float() * count[:, None]).to(torch.bfloat16))         # equal terms: exact but for the last rounding
    buf.check_device_status()


def test_large_rows_on_a_handle():
    """Rows of whole KB, seven a token and more, larger than the memory-side cache: five workgroups a CU, six without a handle."""
    import deep_ep
    T, H, E, R, K = 7507, 4096, 256, 32, 8
    assert shape(move("bf16", T, H, E, R, K)) == (1, 6, 1) and shape(move("bf16", T, H, E, R, K, cached=True)) == (1, 5, 1)
    small = rc.small("handle", T, 16, E, R, K, seed=64, masked_ratio=0.01)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(65), device="cuda", dtype=torch.bfloat16)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    recv, _, _, handle, _ = buf.dispatch(x, small.topk_idx.cuda(), small.topk_weights.cuda(), num_experts=E)
    tokens = handle.recv_src_metadata[:, 0].long()
    assert 7.0 * T < tokens.numel() and torch.equal(recv.view(torch.int16), x[tokens].view(torch.int16))
    again = buf.dispatch(-x, topk_weights=small.topk_weights.cuda(), handle=handle)[0]
    assert torch.equal(again.view(torch.int16), (-x)[tokens].view(torch.int16))
    buf.check_device_status()


@pytest.mark.parametrize("T,H,R,K,chosen", [(5003, 7168, 4, 4, (1, 0, 0)), (5003, 7168, 8, 4, (1, 0, 1)), (9001, 3968, 8, 3, (2, 3, 0)), (292, 7168, 8, 8, (1, 0, 0)), (293, 7168, 8, 8, (2, 0, 0)), (311, 7168, 8, 8, (2, 0, 0))])
def test_v1_rows_of_a_mask(T, H, R, K, chosen):
    """V1 calls without top-k tensors, whose routing lanes are ranks, and the same on their handle."""
    import deep_ep
    idx = rc.small("mask", T, 16, 64, R, K, seed=66).topk_idx
    mask = oracle.layout(idx, 64, R)[2]
    source = torch.cat([torch.nonzero(mask[:, r])[:, 0] for r in range(R)]).cuda()
    assert shape(v1_move("bf16", T, H, R, source.numel())) == chosen
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(67), device="cuda", dtype=torch.bfloat16)
    buf = deep_ep.Buffer(deep_ep.LogicalGroup(0, R))
    per_rank, _, per_expert, mask_d, _ = buf.get_dispatch_layout(idx.cuda(), 64)
    recv, _, _, _, handle, _ = buf.dispatch(x, num_tokens_per_rank=per_rank, is_token_in_rank=mask_d, num_tokens_per_expert=per_expert)
    assert torch.equal(recv.view(torch.int16), x[source].view(torch.int16))
    again = buf.dispatch(-x, handle=handle)[0]
    assert torch.equal(again.view(torch.int16), (-x)[source].view(torch.int16))
    out = buf.combine(recv, handle)[0]
    assert torch.equal(out, (x.float() * mask_d.sum(1).float()[:, None]).to(torch.bfloat16))       # equal terms
    buf.runtime.check_device_status("intranode")
