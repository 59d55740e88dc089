"""BF16 dispatches and combines on both sides of the line up to which rows go through the memory-side cache, in one launch and in two, with
the last column tile of a row partly filled: every received row is the row of its source token, and a combine of the rows as they are is
the token times the number of its rows (exact: at most eight equal terms of seven-bit values)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,R,K,sync", [
    (17700, 2056, 32, 2, 2, True), (18100, 2056, 32, 2, 2, True),         # two launches: 109 and 112 MB of rows, compact
    (5050, 2056, 256, 8, 8, False), (5200, 2056, 256, 8, 8, False),       # one launch
    (19500, 2056, 32, 2, 2, True),                                        # 116 MB returned, compact: the combine's side too
    (13200, 2056, 32, 2, 2, True), (14300, 2056, 32, 2, 2, True),         # expanded, 109 and 118 MB of rows, 103 and 112 returned
    (3250, 2056, 256, 8, 8, False), (3600, 2056, 256, 8, 8, False),       # 107 and 118, 102 and 113
])
@pytest.mark.parametrize("expand", [False, True])
def test_rows_and_sums(T, H, E, R, K, sync, expand):
    import deep_ep
    gen = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randint(-127, 128, (T, H), generator=gen, device="cuda").to(torch.bfloat16) / 16
    w, idx = torch.topk(torch.rand((T, E), generator=gen, device="cuda"), K, dim=1)
    idx = idx.masked_fill(torch.rand((T, K), generator=gen, device="cuda") < 0.05, -1)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K, allow_multiple_reduction=False)
    recv, _, _, handle, _ = buf.dispatch(x, idx, w, num_experts=E, do_cpu_sync=sync, do_expand=expand)
    rank = torch.where(idx >= 0, idx // (E // R), -1)
    per_rank = torch.stack([(rank == r).any(dim=1) for r in range(R)], dim=1)
    n = int(per_rank.sum())
    meta = handle.recv_src_metadata[:n].long()
    if expand:
        lanes = meta[:, 2:]
        rows, tokens = lanes[lanes >= 0], meta[:, :1].expand(-1, K)[lanes >= 0]
        copies = (idx >= 0).sum(dim=1, keepdim=True)
    else:
        rows, tokens, copies = torch.arange(n, device="cuda"), meta[:, 0], per_rank.sum(dim=1, keepdim=True)
    assert rows.numel() == int(copies.sum()) and torch.equal(recv[rows], x[tokens])
    out, _, _ = buf.combine(recv, handle)
    assert torch.equal(out.float(), (x.float() * copies).to(torch.bfloat16).float())
    buf.check_device_status()


@pytest.mark.parametrize("alignment", [280, 288])          # 147 and 151 MB of zeroed rows expected
def test_rows_in_front_of_many_zeroed_ones(alignment):
    import deep_ep
    T, H, E, R, K = 5200, 2056, 256, 8, 8
    gen = torch.Generator(device="cuda").manual_seed(alignment)
    x = torch.randint(-127, 128, (T, H), generator=gen, device="cuda").to(torch.bfloat16) / 16
    w, idx = torch.topk(torch.rand((T, E), generator=gen, device="cuda"), K, dim=1)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K, allow_multiple_reduction=False)
    recv, _, _, handle, _ = buf.dispatch(x, idx, w, num_experts=E, do_expand=True, do_zero_padding=True, expert_alignment=alignment)
    lanes = handle.recv_src_metadata[:, 2:].long()
    rows = lanes[lanes >= 0]
    assert torch.equal(recv[rows], x[handle.recv_src_metadata[:, :1].long().expand(-1, K)[lanes >= 0]])
    recv[rows] = 0
    assert rows.unique().numel() == T * K and not recv.any()
    buf.check_device_status()


# experts with less than one alignment of rows: 235 and 243 MB of rows and padding; with more, 196 and 269; a buffer for more tokens than come
@pytest.mark.parametrize("T,M,E,alignment", [(400, 400, 112, 128), (400, 400, 116, 128), (3000, 3000, 176, 64), (3200, 3200, 160, 128), (400, 4000, 112, 128), (40, 400, 300, 64)])
@pytest.mark.parametrize("sync", [True, False])
def test_rows_among_zeroed_ones(T, M, E, alignment, sync):
    """... and as many rows as fit in the cache, with padding rows that do or do not fit beside them."""
    import deep_ep
    H, R, K = 8208, 4, 2
    gen = torch.Generator(device="cuda").manual_seed(alignment)
    x = torch.randint(-127, 128, (T, H), generator=gen, device="cuda").to(torch.bfloat16) / 16
    w, idx = torch.topk(torch.rand((T, E), generator=gen, device="cuda"), K, dim=1)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=M, hidden=H, num_topk=K, allow_multiple_reduction=False)
    recv, _, _, handle, _ = buf.dispatch(x, idx, w, num_experts=E, do_cpu_sync=sync, do_expand=True, do_zero_padding=True, expert_alignment=alignment)
    n = int(handle.psum_num_recv_tokens_per_scaleup_rank[-1])
    lanes, tokens = handle.recv_src_metadata[:n, 2:].long(), handle.recv_src_metadata[:n, :1].long().expand(-1, K)
    assert int((lanes >= 0).sum()) == T * K and torch.equal(recv[lanes[lanes >= 0]], x[tokens[lanes >= 0]])
    out, _, _ = buf.combine(recv, handle)
    assert torch.equal(out.float(), (x.float() * K).to(torch.bfloat16).float())
    buf.check_device_status()
