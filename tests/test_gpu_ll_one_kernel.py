"""Low-latency dispatch as a single kernel: every workgroup size of it and the two kernels against the oracle on both sides of the lines
between them (which side takes which is in test_launch_lines.py), and a combine through the rows each of them records."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle
from test_gpu_parity import assert_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,T,H,E,K,payload", [
    (8, 384, 4112, 16, 1, "bf16"),         # 3072 tokens, 6144 wavefronts (two tiles a token): 256 threads by its selections
    (8, 385, 4112, 16, 1, "bf16"),         # 3080: two kernels
    (4, 512, 1152, 16, 2, "fp8"),          # 4096 selections: 256
    (4, 513, 1152, 16, 2, "fp8"),          # 4104: 512
    (8, 256, 4112, 16, 4, "bf16"),         # 8192 selections, 4096 wavefronts: 512
    (8, 257, 4112, 16, 4, "bf16"),         # 8224, 4112: two kernels
    (8, 256, 4608, 16, 5, "ue8m0"),        # 10240 selections, 4096 wavefronts, FP8: 1024
    (8, 256, 4224, 16, 8, "fp8"),          # 16384: 1024
    (8, 256, 4224, 16, 9, "fp8"),          # 18432: two kernels
    (8, 257, 2064, 16, 7, "bf16"),         # 4112 wavefronts: two kernels
    (8, 257, 2048, 16, 7, "bf16"),         # 2056: 1024
    (8, 384, 512, 16, 8, "fp8"),           # 24576 selections: 1024
    (8, 384, 512, 16, 9, "fp8"),           # 27648: 1024
    (8, 256, 512, 16, 10, "bf16"),         # 2048 wavefronts: 512 up to 24576 selections
    (8, 256, 512, 16, 13, "bf16"),         # 26624: 1024
    (8, 385, 4112, 16, 2, "bf16"),         # 3080 tokens: two kernels
    (8, 384, 4112, 16, 2, "bf16"),         # 6144 selections, 6144 wavefronts: 512
    (8, 192, 4112, 16, 6, "bf16"),         # 3072 wavefronts: 1024
    (8, 384, 512, 64, 32, "fp8"),          # 98304 selections: 1024
], ids=lambda v: str(v))
def test_single_kernel_lines(R, T, H, E, K, payload):
    import deep_ep
    x, idx, w = rc.c5_sources(seed=23, R=R, T=T, H=H, E=E, K=K)
    idx = idx.masked_fill(torch.rand(idx.shape, generator=torch.Generator().manual_seed(5)) < 0.1, -1)
    fp8, ue8m0 = payload != "bf16", payload == "ue8m0"
    M = -(-T // 4) * 4
    dst = R - 1
    buf = deep_ep.Buffer(deep_ep.LogicalGroup(dst, R), low_latency_mode=True)
    px, ps, cnt, info, rng = oracle.ll_dispatch(list(x), list(idx), M, E, R, dst, fp8, round_scale=ue8m0)
    y = torch.zeros((E // R, R * M, H), dtype=torch.bfloat16)
    for e in range(E // R):
        y[e, :int(cnt[e])] = torch.randn((int(cnt[e]), H), generator=torch.Generator().manual_seed(e)).to(torch.bfloat16)
    back = [oracle.ll_combine(y, idx[s], w[s], info, rng, s, E, R, dst) for s in range(R)]
    x, idx, w, y = x.cuda(), idx.cuda(), w.cuda(), y.cuda()
    for form in ("as it comes", 256, 512, 1024, "two kernels"):
        deep_ep.tuning.ll_threads, deep_ep.tuning.ll_two_kernels = form if isinstance(form, int) else 0, int(form == "two kernels")
        try:
            recv, count, handle, _, _ = buf.low_latency_dispatch(x, idx, M, E, use_fp8=fp8, round_scale=ue8m0, use_ue8m0=ue8m0)
        finally:
            deep_ep.tuning.ll_threads = deep_ep.tuning.ll_two_kernels = 0
        assert_equal(count, cnt, f"packed_recv_count, {form}")
        assert_equal(handle[1], rng, f"packed_recv_layout_range, {form}")
        got = recv[0] if fp8 else recv
        for e in range(E // R):
            n = int(cnt[e])
            assert_equal(handle[0][e, :n], info[e, :n], f"src_info[{e}], {form}")
            assert_equal(got[e, :n], px[e, :n], f"packed_recv_x[{e}], {form}")
            if fp8:
                assert_equal(recv[1][e, :n], oracle.pack_ue8m0(ps[e, :n]) if ue8m0 else ps[e, :n], f"scales[{e}], {form}")
        out, _, _ = buf.low_latency_combine(y, idx, w, handle)
        for s in range(R):
            assert_equal(out[s] + 0.0, back[s] + 0.0, f"combined from source {s}, {form}")


@pytest.mark.parametrize("H,payload", [(4112, "bf16"), (4608, "ue8m0")])
@pytest.mark.parametrize("which", ["none", "last", "every_third", "all"])
def test_single_kernel_reads_the_tokens_that_stay(which, H, payload):
    """Payloads of tokens without a local expert are not read: destinations no token, one, some and every token goes to, the others' rows
    NaN.  The combine goes through the rows the dispatch recorded."""
    import deep_ep
    R, T, E, K, M, dst = 3, 37, 12, 3, 40, 1
    x, idx, w = rc.c5_sources(seed=29, R=R, T=T, H=H, E=E, K=K)
    E_l = E // R
    token = torch.arange(R * T).view(R, T, 1)
    stays = {"none": token < 0, "last": token == R * T - 1, "every_third": token % 3 == 1, "all": token >= 0}[which]
    others = torch.tensor([0, 1, 2, 3, 8, 9, 10, 11])
    away = others[torch.rand((R, T, 8), generator=torch.Generator().manual_seed(2)).argsort(dim=2)[..., :K]]
    here = torch.stack([away[..., 0], dst * E_l + token[..., 0] % E_l, away[..., 2]], dim=2)
    idx = torch.where(stays, here, away)
    x = x.masked_fill(~stays, float("nan"))
    fp8 = payload != "bf16"
    buf = deep_ep.Buffer(deep_ep.LogicalGroup(dst, R), low_latency_mode=True)
    recv, count, handle, _, _ = buf.low_latency_dispatch(x.cuda(), idx.cuda(), M, E, use_fp8=fp8, round_scale=fp8, use_ue8m0=fp8)
    px, ps, cnt, info, rng = oracle.ll_dispatch(list(x), list(idx), M, E, R, dst, fp8, round_scale=fp8)
    assert int(cnt.sum()) == int(stays.sum())
    assert_equal(count, cnt, "packed_recv_count")
    assert_equal(handle[1], rng, "packed_recv_layout_range")
    got = recv[0] if fp8 else recv
    y = torch.zeros((E_l, R * M, H), dtype=torch.bfloat16)
    for e in range(E_l):
        n = int(cnt[e])
        assert_equal(handle[0][e, :n], info[e, :n], f"src_info[{e}]")
        assert_equal(got[e, :n], px[e, :n], f"packed_recv_x[{e}]")
        if fp8:
            assert_equal(recv[1][e, :n], oracle.pack_ue8m0(ps[e, :n]), f"scales[{e}]")
        y[e, :n] = torch.randn((n, H), generator=torch.Generator().manual_seed(e)).to(torch.bfloat16)
    out, _, _ = buf.low_latency_combine(y.cuda(), idx.cuda(), w.cuda(), handle)
    for s in range(R):
        assert_equal(out[s] + 0.0, oracle.ll_combine(y, idx[s], w[s], info, rng, s, E, R, dst) + 0.0, f"combined from source {s}")
