"""Exact-size dispatches on either side of the size up to which outputs are allocated at their bound (64 MiB in all) before the
counts are known: the tensors have the exact number of rows, are contiguous, hold the tokens they should, and past that size no
memory beyond a fifteenth more."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle

pytestmark = pytest.mark.gpu

SHAPES = {"at_the_limit": (507, 8192, 8), "past_the_limit": (509, 8192, 8), "far_past_the_limit": (2049, 8192, 8), "one_token": (1, 1024, 8), "one_rank": (300, 1024, 1)}


@pytest.mark.parametrize("surface", ["elastic", "legacy"])
@pytest.mark.parametrize("shape", SHAPES)
def test_exact_rows(shape, surface):
    import deep_ep
    T, H, R = SHAPES[shape]
    E, K = 64, 8
    small = rc.small(shape, T, 16, E, R, K, seed=60, masked_ratio=0.1)
    ref = oracle.dispatch(small.x, small.topk_idx, small.topk_weights, E, R, 0, T)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(61), device="cuda", dtype=torch.bfloat16)
    idx, w = small.topk_idx.cuda(), small.topk_weights.cuda()
    group = deep_ep.LogicalGroup(0, R)
    for _ in range(2):
        if surface == "elastic":
            buf = deep_ep.ElasticBuffer(group, num_max_tokens_per_rank=T, hidden=H, num_topk=K)
            recv_x, recv_idx, recv_w, handle, _ = buf.dispatch(x, idx, w, num_experts=E)
            tokens, per_expert = handle.recv_src_metadata[:, 0].long(), handle.num_recv_tokens_per_expert_list
            assert handle.num_recv_tokens == ref.num_recv_tokens
            assert torch.equal(recv_w.cpu(), ref.recv_topk_weights)
        else:
            buf = deep_ep.Buffer(group)
            per_rank, _, counts, in_rank, _ = buf.get_dispatch_layout(idx, E)
            recv_x, recv_idx, recv_w, per_expert, handle, _ = buf.dispatch(
                x, num_tokens_per_rank=per_rank, is_token_in_rank=in_rank, num_tokens_per_expert=counts, topk_idx=idx, topk_weights=w)
            tokens = handle[3].long()
        assert recv_x.shape == (ref.num_recv_tokens, H) and recv_x.is_contiguous()
        assert recv_idx.shape == recv_w.shape == (ref.num_recv_tokens, K) and recv_idx.is_contiguous() and recv_w.is_contiguous()
        assert torch.equal(recv_idx.cpu(), ref.recv_topk_idx)
        assert list(per_expert) == ref.num_unaligned_recv_tokens_per_expert.tolist()
        assert torch.equal(tokens.cpu().int(), ref.recv_src_metadata[:, 0])
        assert torch.equal(recv_x, x[tokens])


# T, H, R, K, FP8: rows of 776 bytes of which the payload is 256, so that 4096 x 32 of them pass the limit by what travels beside
# it; and whole rows, FP8 with scales and BF16
MASKED = {"narrow_rows": (4096, 128, 32, 32, False), "fp8_rows": (4096, 7168, 8, 8, True), "bf16_rows": (2049, 7168, 8, 8, False),
          "small": (300, 7168, 8, 8, True)}


@pytest.mark.parametrize("surface", ["elastic", "legacy"])
@pytest.mark.parametrize("shape", MASKED)
def test_memory_kept_with_mostly_masked_routing(shape, surface):
    import deep_ep
    from deep_ep.utils.math import per_token_cast_to_fp8
    T, H, R, K, fp8 = MASKED[shape]
    E = 64
    case = rc.small(shape, T, H, E, R, K, seed=62, masked_ratio=0.97)
    x, idx, w = case.x.cuda(), case.topk_idx.cuda(), case.topk_weights.cuda()
    payload = per_token_cast_to_fp8(x) if fp8 else x
    if surface == "elastic":
        buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
        recv, recv_idx, recv_w, handle, _ = buf.dispatch(payload, idx, w, num_experts=E)
        records = handle.recv_src_metadata
    else:
        buf = deep_ep.Buffer(deep_ep.LogicalGroup(0, R))
        per_rank, _, counts, in_rank, _ = buf.get_dispatch_layout(idx, E)
        recv, recv_idx, recv_w, _, handle, _ = buf.dispatch(payload, num_tokens_per_rank=per_rank, is_token_in_rank=in_rank,
                                                            num_tokens_per_expert=counts, topk_idx=idx, topk_weights=w)
        records = handle[3]
    tensors = [*(recv if fp8 else (recv,)), recv_idx, recv_w, records]
    kept = sum({t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for t in tensors}.values())
    needed = sum(t.numel() * t.element_size() for t in tensors)
    assert kept <= (64 << 20)
    if shape != "small":
        assert kept <= needed + 256 * len(tensors)


# T, H, R, K: both sides of the limit
SIZES = {"up_front": (300, 1024, 8, 6), "afterwards": (1500, 7168, 8, 6)}


def _call(buf, payload, idx, w, E, on_stream=False, **kw):
    """One exact-size dispatch on either surface: rows, scales, indices, weights, source tokens."""
    import deep_ep
    legacy = isinstance(buf, deep_ep.Buffer)
    if on_stream:
        kw.update(previous_event=buf.capture(), allocate_on_comm_stream=True, **{"async_finish" if legacy else "async_with_compute_stream": True})
    if legacy:
        per_rank, _, counts, in_rank, _ = buf.get_dispatch_layout(idx, E)
        if on_stream:
            kw["previous_event"] = buf.capture()
        recv, recv_idx, recv_w, _, handle, event = buf.dispatch(payload, num_tokens_per_rank=per_rank, is_token_in_rank=in_rank,
                                                                num_tokens_per_expert=counts, topk_idx=idx, topk_weights=w, **kw)
    else:
        recv, recv_idx, recv_w, handle, event = buf.dispatch(payload, idx, w, num_experts=E, **kw)
    if on_stream:
        event.current_stream_wait()
    tokens = handle[3] if legacy else handle.recv_src_metadata[:, 0]
    return (*(recv if isinstance(recv, tuple) else (recv, None)), recv_idx, recv_w, tokens.long())


@pytest.mark.parametrize("on_stream", [False, True])
@pytest.mark.parametrize("form", ["elastic_pair", "elastic_cast", "elastic_column_major", "legacy_pair"])
@pytest.mark.parametrize("size", SIZES)
def test_exact_scales(size, form, on_stream):
    import deep_ep
    from deep_ep.utils.math import per_token_cast_to_fp8
    T, H, R, K = SIZES[size]
    E = 64
    small = rc.small(size, T, 16, E, R, K, seed=63, masked_ratio=0.2)
    ref = oracle.dispatch(small.x, small.topk_idx, small.topk_weights, E, R, 0, T)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(64), device="cuda", dtype=torch.bfloat16)
    q, sf = per_token_cast_to_fp8(x)
    idx, w = small.topk_idx.cuda(), small.topk_weights.cuda()
    group = deep_ep.LogicalGroup(0, R)
    buf = deep_ep.Buffer(group) if form == "legacy_pair" else deep_ep.ElasticBuffer(group, num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    kw = {"elastic_cast": dict(cast_to_fp8=True), "elastic_column_major": dict(cast_to_fp8=True, use_tma_aligned_col_major_sf=True)}.get(form, {})
    for _ in range(2):
        recv, recv_sf, recv_idx, _, tokens = _call(buf, (q, sf) if form.endswith("pair") else x, idx, w, E, on_stream, **kw)
        assert recv.shape == (ref.num_recv_tokens, H) and recv_sf.shape == (ref.num_recv_tokens, H // 128)
        assert recv_sf.is_contiguous() == (form != "elastic_column_major")
        assert torch.equal(tokens.cpu().int(), ref.recv_src_metadata[:, 0]) and torch.equal(recv_idx.cpu(), ref.recv_topk_idx)
        assert torch.equal(recv.view(torch.uint8), q[tokens].view(torch.uint8)) and torch.equal(recv_sf, sf[tokens])


@pytest.mark.parametrize("fault", ["out_of_range", "twice"])
@pytest.mark.parametrize("surface", ["elastic", "legacy"])
@pytest.mark.parametrize("size", SIZES)
def test_bad_routing_raises_and_the_next_call_is_clean(size, surface, fault):
    """Up front the move of the bad routing is queued before its layout's verdict is read."""
    import deep_ep
    T, H, R, K = SIZES[size]
    E = 64
    small = rc.small(size, T, 16, E, R, K, seed=65, masked_ratio=0.2)
    ref = oracle.dispatch(small.x, small.topk_idx, small.topk_weights, E, R, 0, T)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(66), device="cuda", dtype=torch.bfloat16)
    idx, w = small.topk_idx.cuda(), small.topk_weights.cuda()
    group = deep_ep.LogicalGroup(0, R)
    buf = deep_ep.Buffer(group) if surface == "legacy" else deep_ep.ElasticBuffer(group, num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    if surface == "legacy":
        layout = buf.get_dispatch_layout(idx, E)                   # of the good routing: only the dispatch sees the bad one
        call = lambda i: buf.dispatch(x, num_tokens_per_rank=layout[0], is_token_in_rank=layout[3], num_tokens_per_expert=layout[2],
                                      topk_idx=i, topk_weights=w)
    else:
        call = lambda i: buf.dispatch(x, i, w, num_experts=E)
    bad = idx.clone()
    bad[T // 2, 0] = E + 5 if fault == "out_of_range" else 7
    if fault == "twice":
        bad[T // 2, 1] = 7
    with pytest.raises(RuntimeError, match="expert"):
        call(bad)
    recv, recv_idx, recv_w, *_ = call(idx)
    tokens = ref.recv_src_metadata[:, 0].long().cuda()
    assert torch.equal(recv, x[tokens]) and torch.equal(recv_idx.cpu(), ref.recv_topk_idx)


@pytest.mark.parametrize("surface", ["elastic", "legacy"])
@pytest.mark.parametrize("routing", ["even", "spread", "one_rank", "nowhere"])
def test_outputs_allocated_for_even_routing(routing, surface):
    """Past the limit outputs are allocated for evenly chosen experts before the counts are known: kept where those fit (and hold
    at most 16 / 15 of what they need), too few where every token goes to every rank, far too many where all go to one or none."""
    import deep_ep
    T, H, R, E, K = 2049, 4096, 8, 64, 8
    gen = torch.Generator().manual_seed(67)
    idx = torch.stack([torch.randperm(E, generator=gen)[:K] for _ in range(T)])
    if routing == "spread":
        idx = torch.arange(K).mul(E // R).add(torch.randint(0, E // R, (T, K), generator=gen))
    elif routing == "one_rank":
        idx = torch.stack([torch.randperm(E // R, generator=gen)[:K] for _ in range(T)]) + 3 * (E // R)
    elif routing == "nowhere":
        idx = torch.full((T, K), -1)
        idx[5, 2] = 9
    w = torch.rand((T, K), generator=gen)
    ref = oracle.dispatch(torch.zeros((T, 16), dtype=torch.bfloat16), idx, w, E, R, 0, T)
    x = torch.randn((T, H), generator=torch.Generator(device="cuda").manual_seed(68), device="cuda", dtype=torch.bfloat16)
    group = deep_ep.LogicalGroup(0, R)
    buf = deep_ep.Buffer(group) if surface == "legacy" else deep_ep.ElasticBuffer(group, num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    for _ in range(2):
        recv, _, recv_idx, recv_w, tokens = _call(buf, x, idx.cuda(), w.cuda(), E)
        assert recv.shape == (ref.num_recv_tokens, H) and recv.is_contiguous()
        assert torch.equal(tokens.cpu().int(), ref.recv_src_metadata[:, 0]) and torch.equal(recv_idx.cpu(), ref.recv_topk_idx)
        assert torch.equal(recv, x[tokens])
        assert recv.untyped_storage().nbytes() * 15 <= recv.numel() * 2 * 16


@pytest.mark.parametrize("surface", ["elastic", "legacy"])
@pytest.mark.parametrize("T", [500, 2049])
def test_memory_for_what_is_received_is_enough(T, surface):
    """Where there is memory for the rows a call receives but not for those it could, it still runs."""
    import deep_ep
    H, R, E, K = 4096, 8, 64, 8
    idx = torch.full((T, K), -1, device="cuda")
    idx[7, 3], idx[T - 1, 0] = 9, 60
    w = torch.ones((T, K), device="cuda")
    x = torch.randn((T, H), device="cuda").to(torch.bfloat16)
    group = deep_ep.LogicalGroup(0, R)
    buf = deep_ep.Buffer(group) if surface == "legacy" else deep_ep.ElasticBuffer(group, num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    for _ in range(2):                                            # what a call keeps exists
        _call(buf, x, idx, w, E)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (12 << 20)) / total)
    try:
        recv, _, recv_idx, recv_w, tokens = _call(buf, x, idx, w, E)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert tokens.tolist() == [7, T - 1] and torch.equal(recv, x[tokens]) and recv_idx.shape == recv_w.shape == (2, K)
    buf_status = getattr(buf, "check_device_status", None)
    if buf_status is not None:
        buf_status()
