"""Combine on both sides of the lines between its column tiles (compact, expanded and V1 rows; few and many rows a token): the same bits
as with either tile forced.  Rows are summed per channel, so the tile must not show; the sums themselves are compared with the oracle
elsewhere.  Low-latency combines likewise, at the lines of tokens and of rows a token."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,T,H,E,R,K", [
    ("compact", 1500, 4096, 8, 2, 2), ("compact", 1536, 4096, 8, 2, 2),            # few rows: 12288 wavefronts of 1 KB
    ("compact", 1195, 3064, 72, 6, 9), ("compact", 1194, 3064, 72, 6, 9),          # many: past seven eighths of 8192
    ("expanded", 512, 4096, 8, 2, 2), ("expanded", 511, 4096, 8, 2, 2),            # 4096
    ("expanded", 1025, 2040, 64, 4, 4), ("expanded", 1024, 2040, 64, 4, 4), ("expanded", 2049, 2048, 64, 4, 4),
    ("compact", 768, 4096, 8, 2, 2), ("compact", 767, 4096, 8, 2, 2),              # few: three quarters of 8192
    ("expanded", 768, 4096, 8, 2, 2), ("expanded", 767, 4096, 8, 2, 2),
    ("compact", 2731, 1536, 8, 2, 2), ("compact", 2730, 1536, 8, 2, 2), ("expanded", 2731, 1536, 8, 2, 2),       # 3 KB rows: a round
    ("v1", 1025, 4096, 64, 8, 2), ("v1", 1024, 4096, 64, 8, 2),                    # a round
    ("v1", 2048, 1024, 64, 8, 8), ("v1", 2047, 1024, 64, 8, 8), ("v1", 1, 520, 64, 8, 8),
])
def test_the_tile_does_not_show(layout, T, H, E, R, K):
    import deep_ep
    gen = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((T, H), generator=gen, device="cuda", dtype=torch.bfloat16)
    bias = torch.randn((T, H), generator=gen, device="cuda", dtype=torch.bfloat16)
    w, idx = torch.topk(torch.rand((T, E), generator=gen, device="cuda"), K, dim=1)
    idx = idx.masked_fill(torch.rand((T, K), generator=gen, device="cuda") < 0.1, -1)
    if layout == "v1":
        buf = deep_ep.Buffer(deep_ep.LogicalGroup(0, R))
        per_rank, _, per_expert, in_rank, _ = buf.get_dispatch_layout(idx, E)
        recv, _, rw, _, handle, _ = buf.dispatch(x, num_tokens_per_rank=per_rank, is_token_in_rank=in_rank, num_tokens_per_expert=per_expert,
                                                 topk_idx=idx, topk_weights=w)
    else:
        buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
        expand = dict(do_expand=True, do_zero_padding=True, expert_alignment=16) if layout == "expanded" else {}
        recv, _, rw, handle, _ = buf.dispatch(x, idx, w, num_experts=E, **expand)
    results = []
    for vecs in (0, 1, 2):
        deep_ep.tuning.combine_vecs = vecs
        try:
            results.append(buf.combine(recv, handle, topk_weights=rw, bias=bias)[:2])
        finally:
            deep_ep.tuning.combine_vecs = 0
    for out, out_w in results[1:]:
        assert torch.equal(out.view(torch.int16), results[0][0].view(torch.int16)) and torch.equal(out_w, results[0][1])


@pytest.mark.parametrize("R,T,H,E,K", [
    (8, 513, 4112, 64, 1), (8, 512, 4112, 64, 1),          # an eighth of a row a token: past 4096 tokens
    (16, 300, 1040, 32, 2), (16, 300, 512, 32, 2),         # ... of 2080 and 1024 bytes
    (8, 520, 7168, 32, 2), (8, 520, 5120, 32, 2),          # a quarter: a seventh and a fifth of 4 KB tiles idle
    (8, 520, 4096, 32, 3),                                 # more
])
def test_the_tile_of_a_low_latency_combine_does_not_show(R, T, H, E, K):
    import deep_ep
    gen = torch.Generator(device="cuda").manual_seed(H)
    x = torch.randn((R, T, H), generator=gen, device="cuda", dtype=torch.bfloat16)
    w, idx = torch.topk(torch.rand((R, T, E), generator=gen, device="cuda"), K, dim=2)
    buf = deep_ep.Buffer(deep_ep.LogicalGroup(R // 2, R), low_latency_mode=True)
    recv, _, handle, _, _ = buf.low_latency_dispatch(x, idx, T, E, use_fp8=False)
    results = []
    for vecs in (0, 1, 2, 4, 7):
        deep_ep.tuning.ll_combine_vecs = vecs
        try:
            results.append(buf.low_latency_combine(recv, idx, w, handle)[0])
        finally:
            deep_ep.tuning.ll_combine_vecs = 0
    mine = (idx // (E // R) == R // 2)
    want = (x.float() * torch.where(mine, w, 0.0).sum(dim=2, keepdim=True))      # every row is its token: K terms, each rounded in fp32 once
    assert torch.allclose(results[0].float(), want, rtol=2 ** -8, atol=0)        # half a BF16 step, and K fp32 roundings
    for out in results[1:]:
        assert torch.equal(out.view(torch.int16), results[0].view(torch.int16))
