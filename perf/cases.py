"""What a program that routes mixture-of-experts tokens has this framework do, as cases that can be timed and compared.

Three kinds of pass, each through the public Python entry points:

  moe      `ElasticBuffer.dispatch` then `.combine`, as one MoE layer of a prefill or training step calls them; with
           `backward` also the two calls of the backward pass (the gradient of a combine is a dispatch with the
           cached handle, the gradient of a dispatch is a combine);
  moe_v1   `Buffer.get_dispatch_layout`, `.dispatch` and `.combine`, the same layer through the V1 surface;
  decode   `Buffer.low_latency_dispatch` then `.low_latency_combine`, one layer of a decode step.

The expert computation between dispatch and combine is the caller's.  With BF16 payloads the received rows go straight
into the combine (experts that do nothing); with FP8 payloads the expert outputs are in the caller's hand already.
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "deepep-ascend_amd"))
import deep_ep  # noqa: E402
from deep_ep.utils.math import per_token_cast_to_fp8  # noqa: E402


def listed():
    return [
        # Decode with one sequence per rank: eight tokens in all, buffers sized for 128 tokens per rank.  Nothing but
        # launches, latency and host work.  BF16 payload.
        dict(name="decode_1", kind="decode", R=8, T=1, M=128, H=7168, E=256, K=8, payload="bf16"),
        # The decode batch low-latency kernels are quoted at: 128 tokens per rank, FP8.
        dict(name="decode_128", kind="decode", R=8, T=128, M=128, H=7168, E=256, K=8, payload="fp8"),
        # A large decode batch with power-of-two scales packed as exponent bytes, as block-scaled FP8 products take them.
        dict(name="decode_512_ue8m0", kind="decode", R=8, T=512, M=512, H=7168, E=256, K=8, payload="ue8m0"),
        # A small model's layer: a call of microseconds with the default exact-size (host-synchronised) dispatch.
        dict(name="small_bf16", kind="moe", T=128, H=1024, E=8, R=2, K=2, payload="bf16", layout="compact", sync=True,
             routing="uniform", backward=False, bias=0, overlap=False),
        # A training micro-batch of a mid-sized model, forward and backward, on the communication stream with events.
        dict(name="train_4096x2048", kind="moe", T=4096, H=2048, E=64, R=8, K=6, payload="bf16", layout="compact", sync=True,
             routing="uniform", backward=True, bias=0, overlap=True),
        # Prefill at the headline shape, FP8 cast fused into the dispatch, exact sizes.
        dict(name="prefill_8192_fp8", kind="moe", T=8192, H=7168, E=256, R=8, K=8, payload="cast", layout="compact", sync=True,
             routing="uniform", backward=False, bias=0, overlap=False),
        # The same batch with skewed routing and masked selections, outputs of worst-case size so that the host never waits.
        dict(name="prefill_skewed_nosync", kind="moe", T=8192, H=7168, E=256, R=8, K=8, payload="cast", layout="compact", sync=False,
             routing="skewed", backward=False, bias=0, overlap=False),
        # Expert-major rows for grouped matrix products: regions padded to 128 rows, column-major scales.
        dict(name="prefill_expanded_128", kind="moe", T=8192, H=7168, E=256, R=8, K=8, payload="cast", layout="expanded", sync=True,
             routing="uniform", backward=False, bias=0, overlap=False),
        # FP8 tokens and scales from the stand-alone cast, moved as they are.
        dict(name="prefill_4096_fp8_pair", kind="moe", T=4096, H=7168, E=256, R=8, K=8, payload="fp8", layout="compact", sync=True,
             routing="uniform", backward=False, bias=0, overlap=False),
        # An odd shape: ragged batch, hidden no multiple of 128 channels, an odd number of selections over six ranks, a residual
        # added in the combine.
        dict(name="odd_1237x2888", kind="moe", T=1237, H=2888, E=72, R=6, K=9, payload="bf16", layout="compact", sync=True,
             routing="uniform", backward=False, bias=1, overlap=False),
        # The V1 calls at the batch their own test uses: 4096 tokens, top-8 of 256.
        dict(name="v1_4096", kind="moe_v1", T=4096, H=7168, E=256, R=8, K=8, payload="bf16", routing="uniform"),
        # The largest: a training micro-batch of 16384 tokens over 32 ranks, forward and backward.
        dict(name="train_16384", kind="moe", T=16384, H=7168, E=256, R=32, K=8, payload="bf16", layout="compact", sync=True,
             routing="uniform", backward=True, bias=0, overlap=False),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "moe_v1", "decode"])
    K = rng.choice([1, 2, 4, 6, 8, 8, 8, 9, 10])
    R = rng.choice([2, 4, 6, 8, 8, 16, 32])
    E = R * rng.choice([1, 2, 4, 8, 12, 16, 32])
    E = min(E, 512 // R * R)
    while E < 2 * K:
        E += R
    if kind == "decode":
        payload = rng.choice(["bf16", "fp8", "fp8", "ue8m0"])
        R = rng.choice([4, 8, 8, 16])
        H = 512 * rng.randint(2, 16)
        T = _log_uniform(rng, 1, 512)
        if payload == "bf16":
            E = max(E // R, 1) * R
            while E < 2 * K:
                E += R
            H += 16 * rng.randint(0, 31)
        else:
            # equally loaded experts: whole rounds of E selections
            K, E = rng.choice([(2, 32), (4, 64), (8, 128), (8, 256), (8, 256)])
            per_round = max(E // (R * K), 1)
            T = max((T + per_round - 1) // per_round, 1) * per_round
        return dict(kind=kind, R=R, T=T, M=max(T, 128), H=H, E=E, K=K, payload=payload)
    T = min(_log_uniform(rng, 32, 16384), 98304 // K)          # no more selections than the largest listed case moves rows
    payload = rng.choice(["bf16", "bf16", "cast", "cast", "fp8"])
    H = 128 * rng.randint(8, 56) if payload != "bf16" else 8 * rng.randint(128, 896)
    if kind == "moe_v1":
        return dict(kind=kind, T=T, H=H, E=E, R=R, K=K, payload="fp8" if payload == "cast" else payload,
                    routing=rng.choice(["uniform", "skewed"]))
    backward = payload == "bf16" and rng.random() < 0.5
    return dict(kind=kind, T=T, H=H, E=E, R=R, K=K, payload=payload, layout=rng.choice(["compact", "compact", "expanded"]),
                sync=rng.random() < 0.7, routing=rng.choice(["uniform", "skewed"]), backward=backward,
                bias=rng.choice([0, 0, 1, 2]), overlap=rng.random() < 0.3)


# ---- routing ----

def _routing(gen, device, T, E, K, how):
    """`topk_idx` [T, K] int64 and `topk_weights` [T, K] fp32.

    uniform   the K best of E independent scores;
    balanced  every run of E / K tokens selects every expert once, in random order (a router held to equal load);
    skewed    popularity falls off like 1 / rank^1.2 over a random order of the experts, one selection in twenty masked (-1).
    """
    if how == "balanced":
        perms = torch.rand((T * K // E, E), generator=gen, device=device).argsort(dim=1)
        idx = perms.view(T, K)[torch.randperm(T, generator=gen, device=device)].contiguous()
        weights = torch.rand((T, K), generator=gen, device=device)
        return idx, weights / weights.sum(dim=1, keepdim=True)
    scores = torch.rand((T, E), generator=gen, device=device)
    if how == "skewed":
        popularity = torch.empty(E, device=device)
        popularity[torch.randperm(E, generator=gen, device=device)] = -1.2 * torch.log(torch.arange(1, E + 1, device=device).float())
        scores = (torch.randn((T, E), generator=gen, device=device) + popularity).softmax(dim=1)
    weights, idx = torch.topk(scores, K, dim=1, sorted=False)
    weights = weights / weights.sum(dim=1, keepdim=True)
    if how == "skewed":
        masked = torch.rand((T, K), generator=gen, device=device) < 0.05
        idx, weights = idx.masked_fill(masked, -1), weights.masked_fill(masked, 0.0)
    return idx.contiguous(), weights.contiguous()


def _shuffled(gen, idx, weights, E, R):
    """Another routing with as many received rows: the tokens in another order, the ranks and the experts of a rank renamed."""
    T, per_rank = idx.shape[0], E // R
    ranks = torch.randperm(R, generator=gen, device=idx.device)
    experts = torch.rand((R, per_rank), generator=gen, device=idx.device).argsort(dim=1)
    renamed = (ranks.unsqueeze(1) * per_rank + experts).flatten()
    order = torch.randperm(T, generator=gen, device=idx.device)
    idx, weights = idx[order], weights[order].contiguous()
    return torch.where(idx >= 0, renamed[idx.clamp(min=0)], -1).contiguous(), weights


def _rows_per_rank(idx, E, R):
    """Tokens that go to each rank, as host numbers."""
    rank = torch.where(idx >= 0, idx // (E // R), -1)
    return [(rank == r).any(dim=1).sum().item() for r in range(R)]


def _align(x, a):
    return (x + a - 1) // a * a


ALIGNMENT = 128          # rows of an expert's region in the expanded layout


def _bf16(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)


# ---- what a program has in hand ----

def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = dict(case)
    R, T, H, E, K = (case[k] for k in "RTHEK")
    if case["kind"] == "decode":
        balanced = case["payload"] != "bf16"
        idx, weights = _routing(gen, "cuda", R * T, E, K, "balanced" if balanced else "uniform")
        state.update(buffer=deep_ep.Buffer(deep_ep.LogicalGroup(0, R), low_latency_mode=True), x=_bf16(gen, R, T, H),
                     idx=idx.view(R, T, K), weights=weights.view(R, T, K))
        if balanced:
            state.update(rows=R * T * K // E, expert_out=_bf16(gen, E // R, R * case["M"], H))
        return state
    # one routing for a case, shuffled by the seed: the sizes of the outputs are the case's
    idx, weights = _routing(torch.Generator(device="cuda").manual_seed(T), "cuda", T, E, K, case["routing"])
    idx, weights = _shuffled(gen, idx, weights, E, R)
    state.update(x=_bf16(gen, T, H), idx=idx, weights=weights)
    if case["kind"] == "moe_v1":
        state["buffer"] = deep_ep.Buffer(deep_ep.LogicalGroup(0, R))
    else:
        state["buffer"] = deep_ep.ElasticBuffer(deep_ep.LogicalGroup(0, R), num_max_tokens_per_rank=T, hidden=H, num_topk=K)
        if case["bias"]:
            biases = tuple(_bf16(gen, T, H) for _ in range(case["bias"]))
            state["biases"] = biases if len(biases) == 2 else biases[0]
        if case["backward"]:
            state["grad_out"] = _bf16(gen, T, H)
    # rows the dispatch returns
    expanded = case.get("layout") == "expanded"
    rows = sum(_rows_per_rank(idx, E, R))
    state["rows"] = rows
    if expanded:
        counts = torch.bincount(idx[idx >= 0], minlength=E).tolist()
        state["expanded_rows"] = sum(_align(c, ALIGNMENT) for c in counts)
    if case["payload"] != "bf16":
        if case.get("sync", True):
            capacity = state["expanded_rows"] if expanded else rows
        else:
            capacity = _align(T * min(K, E) + (ALIGNMENT - 1) * E, ALIGNMENT) if expanded else T * R
        state["expert_out"] = _bf16(gen, capacity, H)
    return state


# ---- one pass ----

def run(state):
    return {"decode": _run_decode, "moe": _run_moe, "moe_v1": _run_moe_v1}[state["kind"]](state)


def _run_decode(s):
    buffer, fp8 = s["buffer"], s["payload"] != "bf16"
    ue8m0 = s["payload"] == "ue8m0"
    recv, count, handle, _, _ = buffer.low_latency_dispatch(s["x"], s["idx"], s["M"], s["E"], use_fp8=fp8, round_scale=ue8m0,
                                                            use_ue8m0=ue8m0)
    combined, _, _ = buffer.low_latency_combine(s["expert_out"] if fp8 else recv, s["idx"], s["weights"], handle)
    if not fp8:
        return combined, count, handle[1]          # every packed row has gone through the combine
    # rows past an expert's count hold nothing; with equal load they are the same rows for every expert
    n = s["rows"]
    return combined, count, handle[1], recv[0][:, :n], recv[1][:, :n], handle[0][:, :n]


def _run_moe(s):
    buffer, expanded, cast = s["buffer"], s["layout"] == "expanded", s["payload"] == "cast"
    overlap = s["overlap"]
    x = per_token_cast_to_fp8(s["x"]) if s["payload"] == "fp8" else s["x"]
    streams = {}
    if overlap:
        streams = dict(previous_event=buffer.capture(), async_with_compute_stream=True, allocate_on_comm_stream=True)
    recv, recv_idx, recv_weights, handle, event = buffer.dispatch(
        x, s["idx"], s["weights"], num_experts=s["E"], expert_alignment=ALIGNMENT if expanded else 1, do_cpu_sync=s["sync"],
        do_expand=expanded, do_zero_padding=expanded, use_tma_aligned_col_major_sf=expanded and s["payload"] != "bf16",
        cast_to_fp8=cast, **streams)
    if overlap:
        event.current_stream_wait()
        streams["previous_event"] = buffer.capture()
    out, out_weights, event = buffer.combine(recv if s["payload"] == "bf16" else s["expert_out"], handle, topk_weights=recv_weights,
                                             bias=s.get("biases"), **streams)
    if overlap:
        event.current_stream_wait()
    outputs = [out, out_weights]
    if s["backward"]:
        if overlap:
            streams["previous_event"] = buffer.capture()
        grad_recv, _, _, _, event = buffer.dispatch(s["grad_out"], handle=handle, do_expand=expanded, **streams)
        if overlap:
            event.current_stream_wait()
            streams["previous_event"] = buffer.capture()
        grad_x, grad_weights, event = buffer.combine(grad_recv, handle, topk_weights=recv_weights, **streams)
        if overlap:
            event.current_stream_wait()
        outputs += [grad_x, grad_weights]
    outputs += [handle.psum_num_recv_tokens_per_scaleup_rank, handle.psum_num_recv_tokens_per_expert,
                handle.num_unaligned_recv_tokens_per_expert, handle.dst_buffer_slot_idx]
    parts = list(recv) if isinstance(recv, tuple) else [recv]
    if s["sync"]:
        return outputs + parts + [recv_idx, recv_weights, handle.recv_src_metadata]
    # outputs of worst-case size: rows past the received ones hold nothing
    n = s["rows"]
    outputs.append(handle.recv_src_metadata[:n])
    return outputs if expanded else outputs + [t[:n] for t in parts + [recv_idx, recv_weights]]


def _run_moe_v1(s):
    buffer = s["buffer"]
    x = per_token_cast_to_fp8(s["x"]) if s["payload"] == "fp8" else s["x"]
    per_rank, _, per_expert, in_rank, _ = buffer.get_dispatch_layout(s["idx"], s["E"])
    recv, recv_idx, recv_weights, per_expert_list, handle, _ = buffer.dispatch(
        x, num_tokens_per_rank=per_rank, is_token_in_rank=in_rank, num_tokens_per_expert=per_expert, topk_idx=s["idx"],
        topk_weights=s["weights"])
    out, out_weights, _ = buffer.combine(recv if s["payload"] == "bf16" else s["expert_out"], handle, topk_weights=recv_weights)
    parts = list(recv) if isinstance(recv, tuple) else [recv]
    return [out, out_weights, *parts, recv_idx, recv_weights, per_rank, per_expert, sum(per_expert_list), *handle]


# ---- what a pass cannot do without ----

def work(case):
    """Every input read once and every output written once, by call; row counts are those of a fixed routing of the case's kind."""
    R, T, H, E, K = (case[k] for k in "RTHEK")
    gen = torch.Generator().manual_seed(0)
    if case["kind"] == "decode":
        tokens, local = R * T, R * T * K / R            # selections that stay on this rank
        row = {"bf16": 2 * H, "fp8": H + H // 128 * 4, "ue8m0": H + H // 128}[case["payload"]]
        dispatch = tokens * H * 2 + tokens * K * 8 + local * (row + 4)
        combine = local * H * 2 + tokens * K * 12 + tokens * H * 2
        return {"bytes": dispatch + combine, "flops": 2 * local * H}
    sample = min(T, 1024)
    idx, _ = _routing(gen, "cpu", sample, E, K, case["routing"])
    rows = sum(_rows_per_rank(idx, E, R)) * T / sample                        # (token, rank) pairs
    selected = (idx >= 0).sum().item() * T / sample                          # (token, expert) pairs
    moved = selected if case.get("layout") == "expanded" else rows
    payload, lists = case["payload"], T * K * 12
    row = 2 * H if payload == "bf16" else H + H // 128 * 4
    row_in = 2 * H if payload in ("bf16", "cast") else row
    placed = rows * (K + 2) * 4 + T * K * 4                                  # the handle's row records and token -> row map
    beside = moved * 4 if case.get("layout") == "expanded" else rows * K * 12
    dispatch = T * row_in + lists + moved * row + beside + placed
    combine = moved * H * 2 + selected * 4 + T * K * 8 + T * H * 2 + T * H * 2 * case.get("bias", 0)
    total = dispatch + combine
    if payload == "fp8":
        total += T * H * 2 + T * row                                         # the stand-alone cast
    if case.get("backward"):
        total += T * H * 2 + moved * H * 2 + T * K * 4 + combine
    if case["kind"] == "moe_v1":
        total += T * K * 8 + T * R                                           # the layout call
    return {"bytes": total, "flops": 2 * moved * H}


def tolerance(case):
    """Rows are moved as bytes, the casts and the order in which a combine adds its rows are fixed by contract (fp32, one
    rounding), and placement follows from the routing alone: every output is reproduced bit for bit."""
    return "exact"
