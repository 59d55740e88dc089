"""The column tiles and residency limits a large move picks by the rows a token goes to and the bytes it writes: calls just
large enough for each of them, ragged batch and ragged hidden, every row checked against the token it came from."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle

pytestmark = pytest.mark.gpu

CASES = {
    "bf16_many_rows_1kb": (3001, 7160, 256, 32, 8, False, False),       # 5 workgroups per CU, 1 KB tiles
    "bf16_few_rows_2kb": (7003, 7160, 64, 4, 4, False, False),          # 2 KB tiles, 4 workgroups per CU
    "cast_many_rows": (3001, 7040, 256, 32, 8, True, False),            # one 1024-channel segment
    "cast_many_rows_small": (37, 2176, 64, 32, 8, True, False),         # ... without a residency limit
    "cast_many_rows_large": (6011, 7040, 256, 32, 8, True, False),      # one segment, four rounds
    "cast_half_empty_segment": (9001, 1152, 256, 32, 8, True, False),   # rows whose second segment would be an eighth full
    "cast_expanded": (2503, 7040, 128, 16, 8, True, True),
    "bf16_two_kb": (25009, 760, 64, 8, 8, False, False),                # whole rows, 5 workgroups per CU
    "bf16_two_kb_many_ranks": (16411, 760, 64, 64, 4, False, False),    # ... and 4, below the size of the other limits
    "bf16_one_kb_many_ranks": (36007, 504, 64, 64, 6, False, False),
    "bf16_two_kb_expanded": (16411, 1024, 64, 8, 8, False, True),       # 1 KB tiles
}


@pytest.mark.parametrize("name", CASES)
def test_every_row_is_its_tokens(name):
    import deep_ep
    from deep_ep.utils.math import per_token_cast_to_fp8
    T, H, E, R, K, cast, expand = CASES[name]
    small = rc.small(name, T, 16, E, R, K, seed=50, masked_ratio=0.05)         # the routing, with a payload of 16 channels
    ref = oracle.dispatch(small.x, small.topk_idx, small.topk_weights, E, R, 0, T, do_expand=expand)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(51), device="cuda", dtype=torch.bfloat16)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    recv, recv_idx, recv_w, handle, _ = buf.dispatch(x, small.topk_idx.cuda(), small.topk_weights.cuda(), num_experts=E, do_expand=expand,
                                                     cast_to_fp8=cast)
    meta = handle.recv_src_metadata
    assert torch.equal(meta.cpu(), ref.recv_src_metadata) and torch.equal(recv_w.cpu(), ref.recv_topk_weights)
    assert torch.equal(handle.dst_buffer_slot_idx.cpu(), ref.dst_buffer_slot_idx)
    tokens = meta[:, 0].long()
    if expand:
        rows = meta[:, 2:]
        tokens = torch.zeros(ref.num_expanded_tokens, dtype=torch.int64, device="cuda").scatter_(
            0, rows[rows >= 0].long(), meta[:, :1].expand_as(rows)[rows >= 0].long())
    else:
        assert torch.equal(recv_idx.cpu(), ref.recv_topk_idx)
    expected = per_token_cast_to_fp8(x) if cast else (x,)
    for got, want in zip(recv if cast else (recv,), expected):
        assert torch.equal(got.view(torch.uint8), want[tokens].view(torch.uint8))
    if not expand:                      # and back: the sum of a token's rows is the token times their number, a power of two or rounded
        y = x[tokens]
        out, _, _ = buf.combine(y, handle)
        count = torch.zeros(T, device="cuda").index_add_(0, tokens, torch.ones(tokens.numel(), device="cuda"))
        assert torch.equal(out, (x.float() * count[:, None]).to(torch.bfloat16))
