"""Padding rows of expanded dispatches, zeroed by workgroups behind the movers of a move on a finished layout, or by a launch behind a single
one: regions that fill an expert's slices unevenly, one slice and many, row-major and column-major scales, scales in blocks on both sides of
their lines, against the oracle on outputs whose memory held other values."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle
from test_gpu_parity import assert_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("payload,T,H,E,R,K,alignment", [
    ("bf16", 1, 8, 2, 1, 1, 2),                  # one padding row of 16 bytes
    ("bf16", 130, 264, 48, 6, 9, 128),           # rows of no whole KB, three slices an expert
    ("bf16", 77, 4104, 5, 1, 2, 700),            # an expert's padding in more than a hundred slices
    ("bf16", 600, 1024, 512, 32, 8, 128),        # slices bounded by the number of experts
    ("bf16", 67, 7168, 256, 8, 8, 128),          # four workgroups a CU, zeroing ones among them
    ("bf16", 67, 7160, 256, 8, 8, 128),          # two
    ("cast", 72, 2560, 128, 16, 8, 128), ("pair", 201, 640, 24, 4, 10, 16),
    ("cast", 1801, 7168, 16, 4, 8, 128), ("cast", 1820, 7168, 16, 4, 8, 128),    # 25.8 and 26.1 MB of input: two launches and one, with blocks
    ("cast", 5499, 3584, 16, 2, 8, 5), ("cast", 5503, 3584, 16, 2, 8, 5),        # 43992 and 44024 rows: columns and blocks
    ("pair", 5182, 5248, 16, 2, 8, 3), ("pair", 5188, 5248, 16, 2, 8, 3),        # a single launch, with blocks
    ("pair", 4146, 5248, 16, 2, 10, 3), ("pair", 4147, 5248, 16, 2, 10, 3),      # 1.6999 and 1.7003 M scales: columns and blocks
], ids=lambda v: str(v))
@pytest.mark.parametrize("columns", [True, False], ids=["columns", "rows"])
def test_padding_rows_read_zero(payload, T, H, E, R, K, alignment, columns):
    import deep_ep
    case = rc.small("padding", T, H, E, R, K, seed=T, masked_ratio=0.03)
    q = case.x if payload == "bf16" else oracle.per_token_cast_to_fp8(case.x)
    ref = oracle.dispatch(q, case.topk_idx, case.topk_weights, E, R, 0, T, expert_alignment=alignment, do_expand=True)
    buf = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
    x = (q[0].cuda(), q[1].cuda()) if payload == "pair" else case.x.cuda()
    layout = dict(do_expand=True, do_zero_padding=True, use_tma_aligned_col_major_sf=columns and payload != "bf16", cast_to_fp8=payload == "cast")
    idx, w, n = case.topk_idx.cuda(), case.topk_weights.cuda(), ref.num_expanded_tokens
    handle = None
    for what in ("exact", "worst-case", "cached"):
        left_behind = [torch.full((size,), 7.0, device="cuda") for size in (n * H // 2 + 1024, n * H // 4 + 1024, 4096)]
        del left_behind
        if what == "cached":
            out, _, rw, _, _ = buf.dispatch(x, topk_weights=w, handle=handle, **layout)
        else:
            out, _, rw, handle_of_call, _ = buf.dispatch(x, idx, w, num_experts=E, expert_alignment=alignment, do_cpu_sync=what == "exact", **layout)
            handle = handle or handle_of_call
        rx, rsf = out if isinstance(out, tuple) else (out, None)
        assert_equal(rx[:n], ref.recv_x, f"recv_x, {what} outputs")
        if rsf is not None:
            assert_equal(rsf[:n], ref.recv_sf, f"recv_sf, {what} outputs")
        assert_equal(rw[:n], ref.recv_topk_weights, f"weights, {what} outputs")
    buf.check_device_status()
