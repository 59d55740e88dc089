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


def combine(T, H, E, R, K, copied, rows=None, expanded=False, meta_rows=None):
    a = _abi.CombineArgs()
    a.num_tokens, a.hidden, a.num_topk, a.num_experts, a.num_ranks, a.num_max_tokens_per_rank, a.do_expand = T, H, K, E, R, T, expanded
    at_once = copied == 2
    a.num_recv_rows = T * R if at_once else int(T * R * (1 - (1 - 1 / R) ** K))
    a.num_x_rows = T * K if expanded else a.num_recv_rows
    a.tuning.rows_copied = copied
    return _abi.lib.deep_ep_hip_combine_tile(ctypes.byref(a))


def v1_combine(T, H, R, K, rows):
    a = _abi.IntranodeCombineArgs()
    a.num_tokens, a.hidden, a.num_ranks, a.num_topk, a.num_x_rows = T, H, R, K, rows
    return _abi.lib.deep_ep_hip_intranode_combine_tile(ctypes.byref(a))


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


# Rows that lie in the caches: the KB a wavefront of the dispatch writes and one of the combine reads.  2 KB wavefronts per CU are T * 7 / 256 for 7168
# channels, T * 4 / 256 for 4096 and T * 3 / 256 for 2888.
SHARED = [
    # T, hidden, experts, ranks, selections, expanded, both phases in one call, KB of both (0: each its own)
    (128, 1024, 8, 2, 2, False, False, 1), (1024, 1024, 64, 8, 4, False, False, 1), (1025, 1024, 64, 8, 4, False, False, 2),      # 4
    (146, 7168, 64, 8, 8, False, False, 1), (147, 7168, 64, 8, 8, False, False, 2),
    (341, 2888, 64, 8, 8, False, False, 1), (342, 2888, 64, 8, 8, False, False, 2),
    (384, 4096, 64, 8, 8, False, False, 1), (385, 4096, 64, 8, 8, False, False, 2),                                               # whole 8 KB: 6
    (548, 7168, 64, 8, 8, True, False, 1), (549, 7168, 64, 8, 8, True, False, 2),                                                 # eight rows: 15
    (1097, 7168, 64, 8, 4, False, False, 2), (1098, 7168, 64, 8, 4, False, False, 0),                                             # 30
    (1, 7168, 64, 8, 8, False, True, 2), (804, 7168, 64, 8, 8, False, True, 2),                                                   # 22
    (292, 7168, 256, 32, 8, False, True, 2), (256, 4096, 64, 8, 8, False, True, 2), (257, 4096, 64, 8, 8, False, True, 1),
    (384, 4096, 64, 8, 8, False, True, 1), (385, 4096, 64, 8, 8, False, True, 2),                                                 # 4 and 6
    (146, 7168, 64, 8, 8, True, True, 1), (147, 7168, 64, 8, 8, True, True, 2),
    (2362, 1064, 64, 8, 8, False, False, 1), (2562, 1064, 64, 8, 4, False, False, 0),                                             # 2128 of 4096 bytes
]


@pytest.mark.parametrize("T,H,E,R,K,expanded,at_once,kb", SHARED)
def test_dispatch_and_combine_share_a_tile(T, H, E, R, K, expanded, at_once, kb):
    s = move("bf16", T, H, E, R, K, expanded=expanded, single=at_once)
    assert s.cached_side == ROWS and s.single_launch == at_once
    both = combine(T, H, E, R, K, 2 if at_once else 1, expanded=expanded)
    own = combine(T, H, E, R, K, 0, expanded=expanded)
    if kb:
        assert s.tile == both == kb
    else:
        assert both == own
    if R == 8 and K >= 4 and T * ((H + 1023) // 1024) < 18 * 256:
        assert own == 1                                   # behind FP8 rows, and for handles that do not say


def test_past_the_line_of_a_single_launch():
    """805 x 7168: 22 a CU.  The move has its own tile; the combine and a dispatch on the handle share that of two launches."""
    a = (805, 7168, 64, 8, 8)
    assert move("bf16", *a, single=True).tile == 4 and combine(*a, 2) == move("bf16", *a, cached=True, rows_copied=2).tile == 2
    b = (2370, 1264, 64, 4, 5)                            # a fourth of the 2 KB tiles empty, 1 KB
    assert move("bf16", *b, expanded=True, cached=True, rows_copied=2).tile == combine(*b, 2, expanded=True) == 1


def test_combine_of_rows_no_bf16_dispatch_wrote():
    assert combine(1535, 2888, 64, 8, 8, 0) == 1 and combine(1536, 2888, 64, 8, 8, 0) == 2                  # 18 a CU
    assert combine(2561, 2888, 64, 8, 4, 0) == 1                                                          # 30


def test_cached_dispatch_has_the_tile_of_the_handle():
    a = (128, 7168, 64, 8, 8)
    assert move("bf16", *a, cached=True).tile == move("bf16", *a, cached=True, rows_copied=1).tile == 1
    assert move("bf16", *a, cached=True, rows_copied=2).tile == move("bf16", *a, single=True).tile == combine(*a, 2) == 2
    assert move("bf16", 1000, 2048, 64, 8, 9, cached=True, rows_copied=2).tile == 2             # top-9 has no single launch: 8 a CU
    assert move("bf16", 100, 7168, 64, 8, 8, expanded=True, alignment=16, pads=True, cached=True, rows_copied=2).tile == 1


def test_v1_tiles():
    for T, rows, kb in ((146, 700, 1), (292, 1400, 1), (293, 1400, 2), (1097, 5000, 2), (1098, 3000, 1), (100, 800, 2)):      # 8 and 30; a row for every rank
        assert v1_combine(T, 7168, 8, 4, rows) == kb
    assert v1_combine(146, 7168, 8, 0, 700) == v1_move("bf16", 146, 7168, 8, 700).tile == 1
    assert v1_combine(292, 7168, 8, 0, 1400) == v1_move("bf16", 292, 7168, 8, 1400).tile == 1
    assert v1_combine(293, 7168, 8, 0, 1400) == v1_move("bf16", 293, 7168, 8, 1400).tile == 2


def test_large_expanded_rows_of_no_whole_kb():
    assert shape(move("bf16", 4927, 5080, 72, 8, 9, expanded=True)) == (1, 2, 0)            # 450.6 MB
    assert shape(move("bf16", 4900, 5080, 72, 8, 9, expanded=True)) == (2, 2, 0)            # 448.1
    assert shape(move("bf16", 9854, 5080, 72, 8, 8, expanded=True))[:1] == (2,)             # eight rows, 801 MB
    assert shape(move("bf16", 4927, 5088, 72, 8, 9, expanded=True)) == (2, 2, 0)            # whole 64 bytes
    assert shape(move("bf16", 4927, 5080, 288, 32, 9, expanded=True)) == (2, 2, 0)


def test_few_rows_among_much_padding():
    few = dict(expanded=True, alignment=128, pads=True)
    s = move("bf16", 300, 7168, 256, 8, 8, **few)
    assert s.cached_side == NOTHING and shape(s) == (1, 4, 0)                    # 34 MB among 500
    assert shape(move("bf16", 300, 7000, 256, 8, 8, **few)) == (2, 2, 0)


def test_large_casts():
    assert shape(move("cast", 16384, 7168, 256, 32, 8)) == (1, 4, 0)              # 7.2 rows of 7 KB
    assert shape(move("cast", 16384, 7168, 256, 16, 8)) == (2, 4, 0)              # 6.5
    assert shape(move("cast", 16384, 7296, 256, 32, 8)) == (2, 4, 0)
    assert shape(move("cast", 8192, 7168, 256, 8, 6)) == (2, 5, 0)                # 4.4
    assert shape(move("cast", 8192, 7168, 256, 8, 8, expanded=True)) == (2, 3, 0)
    assert shape(move("cast", 5210, 5888, 256, 32, 8)) == (2, 4, 0) and shape(move("cast", 5200, 5888, 256, 32, 8)) == (2, 0, 0)       # 220 MB


def test_large_rows_of_whole_kb():
    a = (16384, 7168, 256, 32, 8)
    assert shape(move("bf16", *a)) == (1, 6, 1) and shape(move("bf16", *a, cached=True)) == (1, 5, 1)                     # 7.2 rows
    assert shape(move("bf16", 16384, 7168, 256, 16, 8, cached=True)) == (1, 6, 1)                                        # 6.5
    assert shape(move("bf16", 8000, 7168, 64, 8, 6)) == (1, 0, 1) and shape(move("bf16", 8000, 7168, 256, 32, 5)) == (1, 6, 1)             # 4.4 and 4.7
    assert shape(move("bf16", 8000, 7168, 256, 64, 5, cached=True)) == (1, 0, 1) and shape(move("bf16", 8000, 7168, 64, 8, 8, cached=True)) == (1, 6, 1)   # 4.8, 5.3
    assert shape(move("bf16", 8000, 7168, 256, 64, 4)) == (2, 3, 0) and shape(move("fp8", 16000, 7168, 256, 64, 4)) == (2, 4, 0)
    assert shape(move("bf16", 8000, 7168, 260, 65, 4)) == (1, 0, 1) and shape(move("fp8", 16000, 7168, 260, 65, 4)) == (1, 0, 1)
    assert shape(move("bf16", 8000, 7168, 256, 64, 4, cached=True)) == (1, 0, 1) and shape(move("fp8", 16000, 7168, 220, 55, 4)) == (1, 0, 1)
    assert shape(move("bf16", 6190, 7168, 256, 64, 4)) == (1, 5, 0) and shape(move("bf16", 6290, 7168, 256, 64, 4)) == (2, 3, 0)             # 347 and 353 MB
    assert shape(move("bf16", 4000, 7168, 256, 32, 8)) == (1, 4, 0) and shape(move("bf16", 4000, 7168, 64, 8, 8)) == (1, 5, 0)      # up to 430 MB
    assert shape(move("bf16", 24000, 4096, 64, 8, 6)) == (2, 3, 0)                                                       # rows of 8 KB, 4.4
    assert shape(move("bf16", 16380, 7168, 256, 16, 4)) == (2, 3, 0) and shape(move("bf16", 14174, 8192, 64, 8, 4)) == (2, 4, 0)    # 3.6 and 3.3
    assert shape(v1_move("bf16", 8192, 7168, 4, 22118)) == (1, 0, 0) and shape(v1_move("bf16", 8192, 7168, 8, 26215)) == (1, 0, 1)  # 2.7 and 3.2, no top-k
    assert shape(move("fp8", 16384, 7168, 256, 32, 8)) == (1, 6, 1) and shape(move("fp8", 8192, 7168, 64, 8, 8)) == (1, 0, 1)
    assert shape(move("fp8", 6301, 3968, 64, 8, 8, expanded=True)) == (4, 0, 0) and shape(move("fp8", 9450, 3968, 64, 8, 8, expanded=True)) == (4, 0, 0)   # 200 and 300 MB
    assert shape(move("fp8", 9453, 3968, 64, 8, 8, expanded=True)) == (2, 3, 0)
    assert shape(move("fp8", 20000, 3968, 64, 8, 6)) == (2, 4, 0) and shape(move("fp8", 17000, 3968, 64, 8, 8, expanded=True)) == (2, 3, 0)


def test_large_rows_of_no_whole_kb():
    assert shape(move("bf16", 16746, 8072, 64, 8, 2)) == (2, 5, 0) and shape(move("bf16", 16746, 8072, 64, 64, 2)) == (2, 4, 0)     # 1.9 and 2.0 rows
    assert shape(move("bf16", 9000, 8008, 64, 8, 1)) == (2, 0, 0)
    assert shape(move("bf16", 10000, 1048, 256, 32, 8)) == (4, 2, 0) and shape(move("bf16", 8000, 2040, 64, 8, 8)) == (4, 2, 0)     # 3 and 4 KB
    assert shape(move("bf16", 2230, 5112, 64, 8, 8)) == (2, 2, 0) and shape(move("bf16", 9000, 5112, 64, 8, 6)) == (2, 3, 0)        # 5.3 rows; 92 MB, 4.4
    assert shape(move("bf16", 4500, 5112, 64, 4, 4)) == (2, 3, 0)                                                                     # 2.7


@pytest.mark.parametrize("payload,T,H,K,blocked", [("cast", 5499, 3584, 8, 0), ("cast", 5501, 3584, 8, 1), ("pair", 4146, 5248, 10, 0), ("pair", 4147, 5248, 10, 1),
                                                   ("pair", 5188, 5120, 10, 0)])
def test_scales_in_blocks(payload, T, H, K, blocked):
    """From 44000 moved rows of a cast on, from 1.7 M scales of FP8 pairs of more than 5120 channels on; column-major scales only."""
    a = dict(expanded=True, alignment=3, pads=True)
    payload = "fp8" if payload == "pair" else payload
    assert move(payload, T, H, 16, 2, K, columns=True, **a).blocked_scales == blocked
    assert move(payload, T, H, 16, 2, K, **a).blocked_scales == 0
