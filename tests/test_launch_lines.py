"""Which dispatches take one launch: both sides of the lines drawn by bytes and by rounds of workgroups, which low-latency dispatches take the
single kernel and in workgroups of how many threads, and GPU results on both sides of
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


PADDED_LINES = [
    # payload, T, hidden, top-k, launches: expanded, padding rows of 64 experts over 8 ranks, aligned to 128, to be zeroed
    ("bf16", 600, 2048, 4, 2), ("bf16", 4000, 4096, 8, 2),
    ("cast", 3173, 4096, 8, 2), ("cast", 3174, 4096, 8, 1),                          # 26 MB of input
    ("cast", 7999, 5000 // 128 * 128, 2, 2), ("cast", 4882, 4096, 4, 2), ("cast", 4883, 4096, 4, 1),      # 80 M channels of rows
    ("cast", 5000, 3968, 8, 2), ("cast", 5000, 4096, 8, 1), ("cast", 8191, 4096, 8, 1), ("cast", 8192, 4096, 8, 2),      # 4096 channels; 64 MB of input
    ("fp8", 6103, 4096, 8, 2), ("fp8", 6104, 4096, 8, 1), ("fp8", 7934, 4096, 8, 1), ("fp8", 7935, 4096, 8, 2),         # 200 and 260 MB of rows
    ("fp8", 15000, 4096, 4, 1), ("fp8", 4000, 4096, 8, 2),
]


@pytest.mark.parametrize("payload,T,H,K,launches", PADDED_LINES)
def test_launches_with_padding_to_zero(payload, T, H, K, launches):
    a = _abi.DispatchArgs()
    a.phases = _abi.PHASE_LAYOUT | _abi.PHASE_MOVE
    a.payload = {"bf16": _abi.PAYLOAD_BF16, "fp8": _abi.PAYLOAD_FP8, "cast": _abi.PAYLOAD_CAST_FP8}[payload]
    a.num_tokens, a.hidden, a.num_topk, a.num_experts, a.num_ranks, a.expert_alignment = T, H, K, 64, 8, 128
    a.do_expand = a.do_zero_padding = 1
    assert _abi.lib.deep_ep_hip_dispatch_kernel_launches(ctypes.byref(a)) == launches
    a.tuning.dispatch_launches = 1
    assert _abi.lib.deep_ep_hip_dispatch_kernel_launches(ctypes.byref(a)) == 1
    a.tuning.dispatch_launches, a.expert_alignment = 0, 1                            # nothing to zero: single but for 64 MB of input
    assert _abi.lib.deep_ep_hip_dispatch_kernel_launches(ctypes.byref(a)) == (2 if T * H * (1 if payload == "fp8" else 2) >= 64 << 20 else 1)


LL_LINES = [
    # source ranks, tokens of each, hidden, top-k, local experts, threads (0: two kernels); 256 compute units
    (8, 512, 512, 1, 32, 0),                                                            # 4096 tokens: past 3072
    (8, 384, 7168, 1, 32, 256), (4, 512, 1152, 2, 4, 256), (4, 513, 1152, 2, 4, 512),   # 4096 selections
    (8, 256, 1024, 12, 4, 512), (8, 256, 1024, 13, 4, 1024),                            # eight wavefronts a unit: 24576
    (8, 192, 1024, 32, 4, 512), (8, 193, 1024, 32, 4, 1024),                            # ... and six
    (8, 257, 512, 3, 4, 512), (8, 257, 512, 4, 4, 1024),                                # twelve: 8192
    (8, 384, 512, 2, 4, 512), (8, 384, 512, 3, 4, 1024), (8, 384, 512, 32, 4, 1024),
    (8, 193, 4112, 3, 4, 512), (8, 193, 4112, 10, 4, 512), (8, 193, 4112, 11, 4, 0),    # 1544 tokens of two wavefronts, sixteen: 16384
    (8, 256, 7168, 8, 32, 512), (8, 256, 7168, 9, 32, 0), (8, 257, 7168, 7, 32, 0),     # 4096 wavefronts, and more: 6144
    (8, 384, 7168, 2, 32, 512), (8, 380, 7168, 3, 32, 0),
    (8, 384, 512, 8, 86, 1024), (8, 384, 512, 8, 88, 0),                                # 33 KB of routing table
    (1, 1, 7168, 1, 32, 0), (1, 2, 7168, 1, 32, 256),                                   # two selections
]


def _ll_threads(S, stride, H, K, E_l, use_fp8=0, **knobs):
    a = _abi.LLDispatchArgs()
    a.num_src_ranks, a.src_token_stride, a.hidden, a.num_topk, a.num_local_experts, a.use_fp8 = S, stride, H, K, E_l, use_fp8
    for k, v in knobs.items():
        setattr(a.tuning, k, v)
    return _abi.lib.deep_ep_hip_ll_dispatch_threads(ctypes.byref(a))


@pytest.mark.parametrize("S,stride,H,K,E_l,threads", LL_LINES)
def test_low_latency_threads(S, stride, H, K, E_l, threads):
    assert _ll_threads(S, stride, H, K, E_l) == threads


def test_low_latency_threads_by_knob_and_errors():
    assert _ll_threads(8, 128, 7168, 8, 32, ll_two_kernels=1) == 0
    assert [_ll_threads(8, 128, 7168, 8, 32, ll_threads=n) for n in (256, 512, 1024, 128)] == [256, 512, 1024, 512]
    assert [_ll_threads(8, 256, 7168, K, 32, use_fp8=1) for K in (4, 5, 8, 9)] == [512, 1024, 1024, 0]       # sixteen: the cast is shared by more
    assert _ll_threads(8, 512, 7168, 8, 32, ll_threads=1024) == 0                       # 4096 tokens take two kernels whatever is asked for
    assert _ll_threads(8, 128, 7168, 33, 32) < 0 and _ll_threads(0, 128, 7168, 8, 32) < 0 and _ll_threads(8, 128, 100, 8, 32) < 0
    assert _abi.lib.deep_ep_hip_ll_dispatch_threads(None) < 0


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
