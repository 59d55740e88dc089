"""Which dispatches take one launch: both sides of the lines drawn by bytes and by rounds of workgroups, and GPU results on both sides of
the two lines against the other way of launching (the ways themselves are compared with the oracle elsewhere)."""
import ctypes

import pytest
import torch

from deep_ep import _abi

LINES = [
    # payload, T, hidden, ranks, top-k, experts, launches
    ("bf16", 16383, 2048, 2, 2, 32, 1), ("bf16", 16384, 2048, 2, 2, 32, 2),          # 64 MB of rows copied as they are
    ("fp8", 16383, 4096, 4, 4, 64, 1), ("fp8", 16384, 4096, 4, 4, 64, 2),
    ("cast", 16384, 2048, 2, 2, 32, 1),                                              # a cast of as much is one launch
    ("cast", 6044, 2048, 8, 8, 256, 1), ("cast", 6045, 2048, 8, 8, 256, 2),          # 1536 residents: 1512 movers beside 24 counters
    ("cast", 7168, 2048, 8, 8, 256, 2), ("cast", 7169, 2048, 8, 8, 256, 1),          # 1792 movers
    ("cast", 6045, 2048, 4, 4, 64, 1),                                               # fewer than four rows a token
]


@pytest.mark.parametrize("payload,T,H,R,K,E,launches", LINES)
def test_launches(payload, T, H, R, K, E, launches):
    a = _abi.DispatchArgs()
    a.phases = _abi.PHASE_LAYOUT | _abi.PHASE_MOVE
    a.payload = {"bf16": _abi.PAYLOAD_BF16, "fp8": _abi.PAYLOAD_FP8, "cast": _abi.PAYLOAD_CAST_FP8}[payload]
    a.num_tokens, a.hidden, a.num_topk, a.num_experts, a.num_ranks, a.expert_alignment = T, H, K, E, R, 1
    assert _abi.lib.deep_ep_hip_dispatch_kernel_launches(ctypes.byref(a)) == launches


@pytest.mark.gpu
@pytest.mark.parametrize("payload,T,H,R,K,E", [("bf16", 16384, 2048, 2, 2, 32), ("cast", 6045, 2048, 8, 8, 256)])
def test_both_ways_place_the_same_rows(payload, T, H, R, K, E):
    import deep_ep
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn((T, H), generator=gen, device="cuda", dtype=torch.bfloat16)
    w, idx = torch.topk(torch.rand((T, E), generator=gen, device="cuda"), K, dim=1)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    results = []
    for way in (0, 1):
        deep_ep.tuning.dispatch_launches = way
        try:
            recv, ri, rw, h, _ = buf.dispatch(x, idx, w, num_experts=E, do_cpu_sync=False, cast_to_fp8=payload == "cast")
        finally:
            deep_ep.tuning.dispatch_launches = 0
        n = int(h.psum_num_recv_tokens_per_scaleup_rank[-1])
        parts = [t[:n] for t in (recv if isinstance(recv, tuple) else (recv,))]
        results.append([p.view(torch.uint8) if p.dtype != torch.float32 else p for p in parts] +
                       [ri[:n], rw[:n], h.recv_src_metadata[:n], h.dst_buffer_slot_idx, h.psum_num_recv_tokens_per_expert])
    assert all(torch.equal(a, b) for a, b in zip(*results))
    buf.check_device_status()


@pytest.mark.gpu
@pytest.mark.parametrize("payload,T,H", [("bf16", 512, 2048), ("bf16", 513, 2048),       # 2048 tiles of 1 KB, and past them
                                         ("bf16", 1280, 2056), ("bf16", 853, 2056),      # 2 KB tiles, the last 16 bytes wide: 2559 and past 2560
                                         ("cast", 292, 7168), ("cast", 293, 7168), ("cast", 3, 16256)])
def test_tiles_of_small_calls_place_the_same_rows(payload, T, H):
    """Exact-size calls that leave the chip half empty take narrow tiles: both sides of the lines against the widest tile."""
    import deep_ep
    gen = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn((T, H), generator=gen, device="cuda", dtype=torch.bfloat16)
    w, idx = torch.topk(torch.rand((T, 32), generator=gen, device="cuda"), 6, dim=1)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, 4), num_max_tokens_per_rank=T, hidden=H, num_topk=6)
    knob, results = "cast_pairs" if payload == "cast" else "copy_vecs", []
    for tile in (0, 4):
        setattr(deep_ep.tuning, knob, tile)
        try:
            recv, ri, rw, h, _ = buf.dispatch(x, idx, w, num_experts=32, cast_to_fp8=payload == "cast")
        finally:
            setattr(deep_ep.tuning, knob, 0)
        parts = recv if isinstance(recv, tuple) else (recv,)
        results.append([p.view(torch.uint8) if p.dtype != torch.float32 else p for p in parts] + [ri, rw, h.recv_src_metadata, h.dst_buffer_slot_idx])
    assert all(torch.equal(a, b) for a, b in zip(*results))
