"""The stand-alone FP8 cast at the edges of its tiles (1024-channel segments, two to a wavefront) and on either side of the
rule that picks the vector kernel: whole 16-channel pieces on 16-byte boundaries."""
import pytest
import torch

import routing_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [16, 112, 128, 1008, 1024, 1040, 2048, 2064, 3072, 7168])
@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "misaligned"])
def test_cast_matches_the_recipe_bit_for_bit(hidden, offset):
    from deep_ep.utils.math import per_token_cast_to_fp8
    tokens = 5
    g = torch.Generator().manual_seed(hidden)
    x = (torch.randn((tokens, hidden), generator=g) * torch.rand((tokens, 1), generator=g) * 8).to(torch.bfloat16)
    x[1, -1], x[2, 0] = 300.0, float("nan")
    x[3] = 0.0
    storage = torch.zeros(tokens * hidden + offset, dtype=torch.bfloat16, device="cuda")
    view = storage[offset:].view(tokens, hidden)
    view.copy_(x)
    q, s = per_token_cast_to_fp8(view)
    q_ref, s_ref = oracle.per_token_cast_to_fp8(x)
    nan = q_ref.to(torch.float32).isnan()
    assert torch.equal(q.cpu().to(torch.float32).isnan(), nan)
    assert torch.equal(q.cpu().view(torch.uint8)[~nan], q_ref.view(torch.uint8)[~nan])
    assert torch.equal(s.cpu().nan_to_num(-1.0), s_ref.nan_to_num(-1.0))
