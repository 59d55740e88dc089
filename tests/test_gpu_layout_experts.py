"""Layout launches on both sides of one and two experts a thread of the publishing workgroup (256 and 512 experts), with odd numbers of
experts (the last thread has one), of the chunks whose totals it keeps (sixteen) and of the (rank, chunk) pairs it takes in one trip (4096),
against the oracle."""
import pytest
import torch

import routing_cases as rc
import routing_oracle as oracle
from test_gpu_parity import _buffer, _check_handle, assert_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,R,K", [
    (256, 256, 8, 4), (1, 257, 1, 4), (256, 257, 1, 4), (257, 264, 8, 9), (256, 511, 7, 5),
    (4096, 512, 16, 3), (4097, 512, 16, 3), (8300, 511, 73, 2),
    (256, 513, 27, 4), (600, 513, 27, 4),
    (3000, 512, 256, 3), (4097, 512, 256, 3),          # 12 and 20 padded chunks of 256 ranks
])
@pytest.mark.parametrize("expand", [False, True])
def test_layout_of_many_experts(T, E, R, K, expand):
    case = rc.small("experts", T, 128, E, R, K, seed=E + T, masked_ratio=0.05)
    buf = _buffer(case)
    x, idx, w = case.x.cuda(), case.topk_idx.cuda(), case.topk_weights.cuda()
    align = 4 if expand else 1
    recv, _, _, handle, _ = buf.dispatch(x, idx, w, num_experts=E, expert_alignment=align, do_expand=expand, do_zero_padding=expand)
    ref = oracle.dispatch(case.x, case.topk_idx, case.topk_weights, E, R, 0, case.M, expert_alignment=align, do_expand=expand)
    assert_equal(recv, ref.recv_x, "recv_x")
    assert handle.num_recv_tokens_per_expert_list == ref.num_recv_tokens_per_expert_list
    _check_handle(handle, ref, case, expand)
    counts = buf.get_dispatch_layout(idx, E)
    of = oracle.layout(case.topk_idx, E, R)
    assert_equal(counts[0], of[0], "num_tokens_per_rank")
    assert_equal(counts[2], of[1], "num_tokens_per_expert")
    buf.check_device_status()
