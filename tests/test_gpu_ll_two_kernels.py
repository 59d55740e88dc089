"""Low-latency dispatch as counting kernel + move kernel against the oracle, at the edges of its counting chunks (256 tokens of a
source), of the chunk totals a wavefront sums at once (64), of the selections it looks up at once (4) and of its column tiles."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle
from test_gpu_parity import assert_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,T,H,E,K,payload", [
    (3, 1, 1024, 6, 2, "bf16"),            # one token a source
    (2, 256, 2064, 8, 4, "bf16"),          # a whole chunk; the last tile of a row holds 16 channels
    (2, 257, 3072, 8, 4, "fp8"),           # one token in the second chunk
    (4, 255, 2560, 16, 8, "ue8m0"),        # last tile half full, two to three selections local
    (1, 300, 512, 32, 20, "ue8m0"),        # every selection local: five rounds of look-ups
    (1, 70, 128, 64, 32, "fp8"),
    (2, 8500, 128, 4, 2, "fp8"),           # 68 chunks
], ids=lambda v: str(v))
def test_two_kernels_match_the_oracle(R, T, H, E, K, payload):
    import deep_ep
    x, idx, w = rc.c5_sources(seed=17, R=R, T=T, H=H, E=E, K=K)
    idx = idx.masked_fill(torch.rand(idx.shape, generator=torch.Generator().manual_seed(3)) < 0.1, -1)
    idx[-1, -1] = -1                       # a token none of whose selections is local anywhere
    fp8, ue8m0 = payload != "bf16", payload == "ue8m0"
    M = -(-T // 4) * 4
    before = deep_ep.tuning.ll_two_kernels
    deep_ep.tuning.ll_two_kernels = 1
    try:
        for dst in sorted({0, R - 1}):
            buf = deep_ep.Buffer(deep_ep.LogicalGroup(dst, R), low_latency_mode=True)
            recv, count, handle, _, _ = buf.low_latency_dispatch(x.cuda(), idx.cuda(), M, E, use_fp8=fp8, round_scale=ue8m0, use_ue8m0=ue8m0)
            px, ps, cnt, info, rng = oracle.ll_dispatch(list(x), list(idx), M, E, R, dst, fp8, round_scale=ue8m0)
            assert_equal(count, cnt, "packed_recv_count")
            assert_equal(handle[1], rng, "packed_recv_layout_range")
            got = recv[0] if fp8 else recv
            for e in range(E // R):
                n = int(cnt[e])
                assert_equal(handle[0][e, :n], info[e, :n], f"src_info[{e}]")
                assert_equal(got[e, :n], px[e, :n], f"packed_recv_x[{e}]")
                if fp8:
                    assert_equal(recv[1][e, :n], oracle.pack_ue8m0(ps[e, :n]) if ue8m0 else ps[e, :n], f"scales[{e}]")
            y = torch.zeros((E // R, R * M, H), dtype=torch.bfloat16)
            for e in range(E // R):
                y[e, :int(cnt[e])] = torch.randn((int(cnt[e]), H), generator=torch.Generator().manual_seed(e)).to(torch.bfloat16)
            out, _, _ = buf.low_latency_combine(y.cuda(), idx.cuda(), w.cuda(), handle)      # through the rows the dispatch recorded
            for s in range(R):
                assert_equal(out[s] + 0.0, oracle.ll_combine(y, idx[s], w[s], info, rng, s, E, R, dst) + 0.0, f"combined from source {s}")
    finally:
        deep_ep.tuning.ll_two_kernels = before
