"""How the library moves rows - launches, column tile, workgroups a CU holds, rows in turn, what goes through the memory-side cache - on both
sides of the lines of its rules, for 256 compute units.  Results on both sides are checked elsewhere."""
import ctypes

import pytest

from deep_ep import _abi

PAYLOADS = {"bf16": _abi.PAYLOAD_BF16, "fp8": _abi.PAYLOAD_FP8, "cast": _abi.PAYLOAD_CAST_FP8}
NOTHING, INPUT, ROWS = 0, 1, 2


def move(payload, T, H, E, R, K, expanded=False, alignment=1, pads=False, single=False, cached=False, columns=False, **knobs):
    """(tile, workgroups per CU, rows in turn) and the rest by name; outputs of worst-case size in single calls, exact by even routing else."""
    a = _abi.DispatchArgs()
    a.phases = _abi.PHASE_MOVE | (_abi.PHASE_LAYOUT if single else 0)
    a.payload, a.cached, a.do_expand, a.do_zero_padding = PAYLOADS[payload], cached, expanded, pads
    a.num_tokens, a.hidden, a.num_topk, a.num_experts, a.num_ranks, a.expert_alignment = T, H, K, E, R, alignment
    a.num_max_tokens_per_rank = T
    a.recv_capacity = T * R if single else int(T * R * (1 - (1 - 1 / R) ** K))
    if expanded:
        a.expanded_capacity = T * min(K, E) + (alignment - 1) * E if single else T * K + E * (alignment - 1) // 2
    if payload != "bf16":
        a.num_sf_packs, a.recv_sf = H // 128, 4096
        a.recv_sf_token_stride, a.recv_sf_hidden_stride = (1, a.expanded_capacity) if columns else (H // 128, 1)
    for k, v in knobs.items():
        setattr(a.tuning, k, v)
    s = _abi.MoveShape()
    assert _abi.lib.deep_ep_hip_dispatch_move_shape(ctypes.byref(a), ctypes.byref(s)) == 0
    return s


def v1_move(payload, T, H, R, rows, cached=False):
    """A V1 dispatch without top-k tensors, of so many rows."""
    a = _abi.IntranodeDispatchArgs()
    a.phases = _abi.PHASE_MOVE
    a.payload, a.cached, a.num_tokens, a.hidden, a.num_ranks, a.recv_capacity = PAYLOADS[payload], cached, T, H, R, rows
    s = _abi.MoveShape()
    assert _abi.lib.deep_ep_hip_intranode_move_shape(ctypes.byref(a), ctypes.byref(s)) == 0
    return s


def shape(s):
    return s.tile, s.workgroups_per_cu, s.rows_in_turn


def test_knobs_are_told_back():
    s = move("bf16", 4096, 4096, 64, 8, 8, copy_vecs=4, move_workgroups_per_cu=3)
    assert shape(s) == (4, 3, 0) and s.cached_side == INPUT
    assert shape(move("cast", 4096, 4096, 64, 8, 8, cast_pairs=7, move_workgroups_per_cu=8)) == (7, 0, 0)
    assert move("cast", 4096, 4096, 64, 8, 8, single=True).single_launch == 1
    assert move("cast", 4096, 4096, 64, 8, 8, single=True, dispatch_launches=2).single_launch == 0
    assert bytes(move("bf16", 0, 4096, 64, 8, 8, single=True)) == bytes(ctypes.sizeof(_abi.MoveShape))
    assert v1_move("bf16", 1000, 4096, 8, 5000).single_launch == 0


def test_errors():
    a, s = _abi.DispatchArgs(), _abi.MoveShape()
    assert _abi.lib.deep_ep_hip_dispatch_move_shape(None, ctypes.byref(s)) < 0
    assert _abi.lib.deep_ep_hip_dispatch_move_shape(ctypes.byref(a), ctypes.byref(s)) < 0           # no experts
    a.num_tokens, a.num_topk, a.num_experts, a.num_ranks, a.hidden, a.payload, a.expert_alignment = 16, 2, 8, 2, 64, 9, 1
    assert _abi.lib.deep_ep_hip_dispatch_move_shape(ctypes.byref(a), ctypes.byref(s)) < 0           # payload
    a.payload, a.hidden = _abi.PAYLOAD_BF16, 0
    assert _abi.lib.deep_ep_hip_dispatch_move_shape(ctypes.byref(a), ctypes.byref(s)) < 0
    assert _abi.lib.deep_ep_hip_intranode_move_shape(ctypes.byref(_abi.IntranodeDispatchArgs()), ctypes.byref(s)) < 0
    assert _abi.lib.deep_ep_hip_combine_tile(ctypes.byref(_abi.CombineArgs())) < 0
    assert _abi.lib.deep_ep_hip_intranode_combine_tile(ctypes.byref(_abi.IntranodeCombineArgs())) < 0


@pytest.mark.parametrize("T,side", [(1916, ROWS), (1917, INPUT), (17857, INPUT), (17858, NOTHING)])
def test_what_the_cache_holds_by_bytes(T, side):
    assert move("bf16", T, 5464 if T < 3000 else 7168, 64, 8, 8).cached_side == side


@pytest.mark.parametrize("E,side", [(128, ROWS), (136, INPUT)])
def test_what_the_cache_holds_among_padding(E, side):
    """400 x 7168 top-8 aligned to 128, in outputs of worst-case size: 46 MB of rows in 235 and 250 MB that are in use."""
    s = move("bf16", 400, 7168, E, 8, 8, expanded=True, alignment=128, single=True)
    assert s.single_launch == 1 and s.cached_side == side
