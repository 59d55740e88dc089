"""Column-major scales of zero-padded expanded dispatches (stored in blocks of 64 rows by the move kernel, put into their columns by the
pad kernel, in large calls) against the oracle: last blocks that are not full, odd and many scales a row, both payloads,
exact, worst-case and cached outputs."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle
from test_gpu_parity import assert_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,R,K,alignment", [
    (2050, 1024, 8, 2, 8, 2),          # two rows a token and expert: few padding rows
    (2048, 1152, 12, 4, 8, 6),         # odd number of scales, regions of 6: blocks start inside padding
    (1100, 2048, 32, 8, 8, 128),       # padding rows fill whole blocks
    (300, 16384, 16, 2, 4, 2),         # as many scales a row as a block may have
    (300, 16512, 16, 2, 4, 2),         # one more: stored into their columns at once
    (2048, 1024, 8, 1, 7, 128),        # narrow rows
    # in blocks from 850000 scales and 14000 rows on, padding rows counted double:
    (1300, 2048, 128, 8, 8, 512),      # padding rows fill whole blocks
    (100, 16384, 128, 2, 4, 128),      # as many scales a row as a block may have, an expert's few rows alone in its region
    (2300, 2944, 64, 4, 6, 400),       # 23 scales: the last trip of a block is not full
    (1803, 7168, 8, 4, 8, 128), (1768, 7168, 8, 4, 8, 128),       # 56 scales: both sides of the line of scales
    (14011, 7808, 8, 4, 1, 2), (13940, 7808, 8, 4, 1, 8),         # 61: both sides of the line of rows, the last block not full
], ids=lambda v: str(v))
@pytest.mark.parametrize("cast", [True, False])
def test_blocked_scales_match_the_oracle(T, H, E, R, K, alignment, cast):
    import deep_ep
    case = rc.small("scale_blocks", T, H, E, R, K, seed=7, masked_ratio=0.07)
    case.topk_idx[case.topk_idx == 1] = -1                    # an expert without rows
    case.topk_weights[case.topk_idx < 0] = 0.0
    q = oracle.per_token_cast_to_fp8(case.x)
    ref = oracle.dispatch(q, case.topk_idx, case.topk_weights, E, R, 0, T, expert_alignment=alignment, do_expand=True)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    x = case.x.cuda() if cast else (q[0].cuda(), q[1].cuda())
    layout = dict(do_expand=True, do_zero_padding=True, use_tma_aligned_col_major_sf=True, cast_to_fp8=cast)
    idx, w, n = case.topk_idx.cuda(), case.topk_weights.cuda(), ref.num_expanded_tokens
    (rx, rsf), _, rw, handle, _ = buf.dispatch(x, idx, w, num_experts=E, expert_alignment=alignment, **layout)
    assert rx.shape[0] == n and rsf.stride() == (1, (n + 3) // 4 * 4)
    (nx, nsf), _, nw, _, _ = buf.dispatch(x, idx, w, num_experts=E, expert_alignment=alignment, do_cpu_sync=False, **layout)
    (cx, csf), _, cw, _, _ = buf.dispatch(x, topk_weights=w, handle=handle, **layout)
    for got_x, got_sf, got_w, what in ((rx, rsf, rw, "exact"), (nx[:n], nsf[:n], nw[:n], "worst-case"), (cx, csf, cw, "cached")):
        assert_equal(got_x, ref.recv_x, f"recv_x, {what} outputs")
        assert_equal(got_sf, ref.recv_sf, f"recv_sf, {what} outputs")
        assert_equal(got_w, ref.recv_topk_weights, f"weights, {what} outputs")
    buf.check_device_status()
