"""Large moves on a finished layout, just past each line of their choice of a column tile and of the workgroups a CU holds: rows that end inside
a vector group, a tile and on one, padded and masked calls, every word against the token it came from."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle

pytestmark = pytest.mark.gpu

CASES = {   # tokens, channels, experts, ranks, selections, payload, expanded, alignment
    "one_kb_by_wavefronts": (1921, 4096, 64, 2, 2, "bf16", False, 1),              # 60 wavefronts of 1 KB per CU
    "wide_by_wavefronts": (1923, 4096, 64, 2, 2, "bf16", False, 1),
    "two_kb_by_wavefronts": (3847, 2040, 64, 8, 6, "bf16", False, 1),
    "ragged_two_workgroups": (2237, 5112, 64, 8, 8, "bf16", False, 1),             # 110 MB of rows
    "ragged_three_workgroups": (3301, 5112, 64, 4, 4, "bf16", False, 1),
    "ragged_three_kb": (10007, 1048, 256, 32, 8, "bf16", False, 1),                # 4 KB tiles, the last vectors of a row absent
    "ragged_four_kb": (8009, 2040, 64, 8, 8, "bf16", False, 1),
    "ragged_two_rows": (9001, 3976, 64, 8, 2, "bf16", False, 1),
    "ragged_two_rows_many_ranks": (9001, 3976, 64, 64, 2, "bf16", False, 1),
    "ragged_one_row": (9001, 8008, 64, 8, 1, "bf16", False, 1),
    "expanded_one_kb": (7507, 2552, 64, 8, 8, "bf16", True, 1),                    # two workgroups per CU, 300 MB
    "expanded_two_kb": (4001, 2552, 64, 8, 8, "bf16", True, 16),
    "whole_five_workgroups": (6607, 2048, 64, 8, 8, "bf16", False, 1),
    "whole_four_workgroups": (6607, 2048, 256, 32, 8, "bf16", False, 1),
    "whole_power_of_two": (10007, 4096, 64, 8, 8, "bf16", False, 1),               # 430 MB
    "whole_few_rows": (9001, 4096, 64, 8, 4, "bf16", False, 1),
    "fp8_four_workgroups": (20011, 3968, 64, 8, 6, "fp8", False, 1),
    "fp8_three_workgroups": (17011, 3968, 64, 8, 8, "fp8", True, 1),
    "cast_five_workgroups": (12007, 4992, 64, 8, 6, "cast", False, 1),
    "cast_four_workgroups": (12007, 4992, 64, 8, 8, "cast", False, 1),
    "cast_three_workgroups": (7001, 4992, 64, 8, 8, "cast", True, 1),
}


@pytest.mark.parametrize("name", CASES)
def test_every_word_is_its_tokens(name):
    import deep_ep
    from deep_ep.utils.math import per_token_cast_to_fp8
    T, H, E, R, K, payload, expand, A = CASES[name]
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


@pytest.mark.parametrize("T,H,E,R,K", [
    (211, 7960, 64, 8, 8), (1, 4096, 8, 4, 2), (7, 2040, 64, 8, 8), (352, 7168, 64, 8, 8), (353, 7168, 64, 8, 8),   # 2 KB; 22 wavefronts of 7168 per CU
    (437, 7168, 256, 32, 8), (439, 7168, 256, 32, 8), (1409, 4096, 64, 8, 4), (1407, 4088, 64, 8, 4),              # 1 KB: 12
])
def test_rows_of_a_single_launch_and_their_sum(T, H, E, R, K):
    import deep_ep
    small = rc.small("single", T, 16, E, R, K, seed=62, masked_ratio=0.05)
    ref = oracle.dispatch(small.x, small.topk_idx, small.topk_weights, E, R, 0, T)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(63), device="cuda", dtype=torch.bfloat16)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    recv, _, w, handle, _ = buf.dispatch(x, small.topk_idx.cuda(), small.topk_weights.cuda(), num_experts=E, do_cpu_sync=False)
    n = ref.recv_src_metadata.shape[0]
    assert torch.equal(handle.recv_src_metadata[:n].cpu(), ref.recv_src_metadata)
    tokens = handle.recv_src_metadata[:n, 0].long()
    assert torch.equal(recv[:n].view(torch.int16), x[tokens].view(torch.int16))
    out, _, _ = buf.combine(recv, handle, topk_weights=w)
    count = torch.zeros(T, device="cuda").index_add_(0, tokens, torch.ones(n, device="cuda"))
    assert torch.equal(out, (x.float() * count[:, None]).to(torch.bfloat16))         # equal terms: exact but for the last rounding
    buf.check_device_status()
