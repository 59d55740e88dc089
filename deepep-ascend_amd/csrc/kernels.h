// Internal interface between the C-ABI entry points (api.hip) and the kernel launchers.
// Parameter blocks are plain structs passed to kernels by value.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

namespace deep_ep_hip {

// Single-launch dispatch: number of completion counters ("gates") the movers spread over, and the distance between
// two of them in 32-bit words (one cache line each).  A persistent move kernel (never part of a single launch) keeps its
// item counter in one of these lines and counts its workgroups out on `gates_finished`; every launch leaves all of them
// at zero.
constexpr int kDispatchGates = 256;
constexpr int kDispatchGateStride = 32;
constexpr int kMaxCountBlocks = 1024;
constexpr int kSingleLaunchTopk = 8;         // selections a token, at most

// Single-launch dispatch: words that counting and publishing workgroups hand to the movers of the same launch carry
// the launch's tag in their upper bits, so that a reader knows a word of this launch from what an earlier launch left
// at the same place and needs no separate flag (and the writer need not wait for its store before it raises one).
// The tagged tables live in the zero-initialised bookkeeping part of the workspace, which only these kernels write:
// every word there is zero, or carries the tag of a launch since the tables were last cleared.  Tags run through
// 1 .. kTagPeriod; the launch that uses the last one clears the tables.
constexpr int kTagShift = 18;
constexpr uint32_t kTagValueMask = (1u << kTagShift) - 1u;
constexpr uint32_t kTagPeriod = (1u << (32 - kTagShift)) - 1u;      // 16383
constexpr int kTaggedRankWords = 1024;       // R x chunks (padded to a multiple of 4)
constexpr int kTaggedExpertWords = 8192;     // chunks x experts (padded to a multiple of 32)
constexpr int kTaggedPosWords = 131072;      // tokens x lanes

// A position word: bits 0-8 the slot of the token inside its chunk for the lane's destination rank (master lanes
// only), bits 9-17 the position of the lane inside its chunk for its expert, kNoPosition = none; a single-launch
// dispatch puts its tag above them.
constexpr uint32_t kNoPosition = 0x1ffu;
constexpr int kExpertPositionShift = 9;

// Byte offsets of the regions carved out of the caller's workspace.
struct WorkspaceLayout {
    size_t status;         // int32: device status bits
    size_t done_counter;   // uint32: workgroups of the layout kernel that have finished
    size_t totals;         // int32[2]: total compact rows, total expanded rows (incl. padding)
    size_t generation;     // uint32: single-launch dispatches since the tagged tables were cleared (tag = generation + 1)
    size_t gates_finished; // uint32: gates whose movers have all read the tagged tables
    size_t chunk_done;     // int32[1024]: per-chunk completion flags of a single-launch dispatch (counting workgroup -> publisher)
    size_t gates;          // uint32[kDispatchGates], one per 128-byte line: movers that have read the tagged tables
    size_t tagged;         // start of the tagged tables; everything before it reads zero between launches but for
                           // status, totals and generation
    size_t tagged_rank;    // uint32[kTaggedRankWords]: rank_counts of the running single-launch dispatch, tagged
    size_t tagged_expert;  // uint32[kTaggedExpertWords]: its expert_bases, tagged
    size_t tagged_expert_counts;   // uint32[kTaggedExpertWords]: expert_counts of an expanded single-launch dispatch, tagged
    size_t tagged_pos;     // uint32[kTaggedPosWords]: its position words, tagged
    size_t tagged_end;
    size_t expert_start;   // int32[E]: first expanded row of each expert
    size_t rank_counts;    // int32[R][C padded to a multiple of 4]: per-chunk totals of the rank buckets, transposed
    size_t rank_bases;     // int32[R][C padded]: first compact row of every (rank, chunk)
    size_t expert_counts;  // int32[C][E padded to a multiple of 32]: per-chunk totals of the expert buckets
    size_t expert_bases;   // int32[C][E padded]: first expanded row of every (chunk, expert)
    size_t pos;            // uint32[Tmax*K]: position words of a dispatch in two launches
    size_t total_bytes;
};

WorkspaceLayout make_workspace_layout(int num_max_tokens, int num_topk, int num_experts, int num_ranks);

// The tables the layout pass leaves in the workspace for the move kernels.  A chunk is 256 consecutive tokens.
//   rank_counts[r][c]    rows chunk c puts into rank r's bucket (transposed: consumers prefix-sum along a row)
//   rank_bases[r][c]     first compact row of (rank r, chunk c) = rows of lower ranks + rows of earlier chunks;
//                        rank_bases[r][0] is the start of rank r's bucket
//   expert_counts[c][e]  rows chunk c puts into expert e's region (one writer per cache line: chunk c's workgroup)
//   expert_bases[c][e]   first expanded row of (chunk c, expert e) = start of the region + rows of earlier chunks
// A row is then "base of (bucket, chunk) + position inside the chunk".
struct LayoutTables {
    int32_t* rank_counts;
    int32_t* rank_bases;
    int32_t* expert_counts;
    int32_t* expert_bases;
    int chunks_padded;    // row length of the rank tables (chunks rounded up to a multiple of 4)
    int experts_padded;   // row length of the expert tables (experts rounded up to a multiple of 32)
};

// Where the public results of the layout computation go (any pointer may be NULL).
struct PublishParams {
    int R, E;
    int A;            // expert alignment
    int do_expand;
    int32_t* num_tokens_per_rank;
    int32_t* num_tokens_per_expert;
    int32_t* psum_rank;
    int32_t* psum_expert;
    int32_t* num_unaligned;
    int32_t* cumulative_stats;
    int32_t* host_counts;            // host-mapped: [R] rank counts, [E] aligned expert counts, then the status word; v as -v-1
    const int32_t* status;           // the device status word (read for host_counts)
    int32_t* expert_start;           // workspace
    int32_t* totals_out;             // workspace: total compact rows, total expanded rows
};

struct LayoutParams {
    const int64_t* topk_idx;
    const uint8_t* route_mask;       // [T, R] bool: when set, lane r of token t is "rank r, if the mask says so" (K = E = R)
    int T, K, E, R, E_l;
    int vec_idx;          // topk_idx is 16-byte aligned (set by the launcher)
    int lds_totals;       // layout kernel of one workgroup: where its totals lie in LDS, bytes (set by the launcher)
    uint8_t* is_token_in_rank;       // optional, layout launch only
    int64_t* copied_topk_idx;        // optional
    PublishParams pub;
    int32_t* status;
    uint32_t* done_counter;
    LayoutTables tab;                // the base tables are optional (layout-only calls have no use for them)
    int expert_bases;                // 1: also tab.expert_bases (expanded layout)
    uint32_t* pos;                   // optional (layout-only calls skip the per-lane positions)
    // Single-launch dispatch (else NULL): chunk totals of the rank buckets go to tagged_rank as well, tagged like the
    // position words, with the tag *generation names when the workgroup starts.
    uint32_t* tagged_rank;
    uint32_t* tagged_expert_counts;  // expanded layout (else NULL): likewise the chunk totals of the expert buckets, for the publisher
    const uint32_t* generation;
};

// The channel matrices of a V1 handle; R = 0: not wanted.
struct IntranodePrefixParams {
    const uint8_t* mask;             // [T, R]
    int T, R, C, rank_idx;
    int32_t* rank_prefix_matrix;         // [R, R]
    int32_t* channel_prefix_matrix;      // [R, C] inclusive over channels
    int32_t* recv_channel_prefix_matrix; // [R, C] exclusive starts
};

// `prefix`, if wanted, rides in the same launch.
hipError_t launch_layout_kernel(const LayoutParams& p, const IntranodePrefixParams& prefix, hipStream_t stream);
hipError_t launch_intranode_prefix(const IntranodePrefixParams& p, hipStream_t stream);

// Alignment padding of an expanded layout: the rows behind the actual ones of every expert.
struct PadParams {
    uint8_t* recv_x;
    uint32_t* recv_sf;
    int64_t rsf_ts, rsf_hs;
    int num_sf_packs;
    float* recv_topk_weights;
    const int32_t* psum_expert;     // start + actual count (expanded convention)
    const int32_t* num_unaligned;
    int64_t expanded_capacity;
    int E, A, out_row_bytes;
    int sf_blocked;                  // recv_sf is in blocks: turned by zero_padding_kernel
    int slices;                      // workgroups that share the padding of an expert (pad_slices)
};

int pad_slices(int experts, int alignment, int out_row_bytes);

struct MoveParams {
    const uint8_t* x;
    const uint32_t* sf;
    int64_t sf_ts, sf_hs;
    int num_sf_packs;
    const int64_t* topk_idx;
    const uint8_t* route_mask;       // see LayoutParams
    const float* topk_weights;
    const uint32_t* pos;
    const int32_t* expert_start;
    const int32_t* cached_slot;
    int32_t* dst_buffer_slot_idx;
    const int32_t* psum_rank;
    int32_t* recv_src_metadata;
    uint8_t* recv_x;
    uint32_t* recv_sf;
    int64_t rsf_ts, rsf_hs;
    int64_t* recv_topk_idx;
    float* recv_topk_weights;
    int64_t recv_capacity, expanded_capacity;
    int T, H, K, E, R, E_l, rank_idx, M;
    float rcp_E_l;       // 1 / E_l (set by the launcher)
    int cached, do_expand;
    int payload;         // DEEP_EP_HIP_PAYLOAD_*
    int row_bytes;       // input row bytes
    int tiles;           // column tiles per token
    int sf_blocked;      // recv_sf is column-major and the pad kernel follows: scales go out in blocks (below)
    int zeroed_rows;     // padding rows this call zeroes, as expected: half an alignment for each expert, or what is
                         // left of one alignment for each where an expert has fewer rows than that
    int v1;              // a V1 call (kb_of_wavefront)
    int like_single;     // a cached handle of a single launch: its tile (kb_of_wavefront)
    int shared_tile;     // the combine has the same tile: workgroups on the XCD of its (set by the launcher)
    int row_by_row;      // a wavefront waits for the stores of a row before it starts the next (set by the launcher)
    unsigned warm_lds_offset;   // single-launch cast: byte offset (in the dynamic LDS) of the 4 KB landing area of the
                                // cache-warming loads, 0 = none
    unsigned warm_ahead;        // ... and how many work items ahead of its own a wavefront warms
    int xcd_remap;       // give each XCD a contiguous token range
    int plain_loads;     // payload loads without the non-temporal hint
    int cast_pairs;      // forced column tile of the fused cast, 0 = choose
    int copy_vecs;       // forced column tile of the pass-through kernels, 0 = choose
    LayoutTables tab;    // written by the layout pass
    PublishParams pub;   // single-launch dispatch: what counting workgroup 0 publishes
    int32_t* status;
    // Single-launch dispatch: the first count_blocks workgroups of the grid count (one 256-token chunk each), the
    // last of them to finish publishes; the movers wait on `sync` before they read any of it.
    int fused;
    int count_blocks;
    unsigned num_movers;     // mover workgroups (set by the launcher)
    int num_cus;             // compute units of the device (set by the launcher)
    LayoutParams lay;        // what the counting workgroups need (lay.pub is unused: `pub` above is published)
    int32_t* chunk_done;     // [kMaxCountBlocks] flags of the counting workgroups for the publisher: totals and positions stored
    uint32_t* gates;         // [kDispatchGates] wrapping counters of the movers that are done reading, kDispatchGateStride words apart
    uint32_t* gates_finished;    // wrapping counter of the gates all of whose movers are done
    unsigned mover_spin_limit;   // reads a mover repeats for a word of the layout before it gives up (set from the tuning block)
    int move_workgroups_per_cu;  // forced residency of a move kernel on a finished layout, 0 = choose (tuning block)
    int warm_rounds;             // rounds ahead the first movers of a single launch warm the caches, 0 = choose, < 0 = none (tuning block)
    int persistent_movers;       // fused-cast move kernel on a finished layout as a persistent kernel with a work queue and this many mover wavefronts per CU, 0 = off (tuning block)
    uint32_t* generation;        // see WorkspaceLayout
    uint32_t* tagged;            // the tagged tables, tagged_words long: cleared by the launch that uses the last tag
    int tagged_words;
    const uint32_t* tagged_rank;
    uint32_t* tagged_expert;
    const uint32_t* tagged_expert_counts;
    // V1 (intranode) conventions
    int rank_lanes;          // routing lanes are ranks (mask routing or a cached send_head), K == R
    int slot_is_row;         // cached_slot holds rows of the receive buffer, not rank * M + slot
    int zero_nonlocal_w;     // weights of lanes routed to another rank are delivered as 0
    int32_t* send_head;      // [T, R] out: receive row of token t on rank r, or -1
    int32_t* recv_src_idx;   // [recv_capacity] out: source token of each receive row
    // A move on a finished layout zeroes the padding too: pad_blocks workgroups behind the movers, 0 = not wanted
    unsigned pad_blocks;
    PadParams pad;
};

hipError_t launch_dispatch_move(MoveParams p, hipStream_t stream);
// What launch_dispatch_move takes for these parameters (p.fused and p.sf_blocked set).
struct MoveChoice {
    int tile;            // KB of row (fused cast: 1024 channels) per wavefront
    int per_cu;          // workgroups a CU holds at a time, 0 = as many as fit
    int in_turn;         // a row's stores are awaited before the next row's
    int cached_side;     // what goes through the memory-side cache: 0 nothing, 1 the input, 2 the rows
};
MoveChoice choose_move(const MoveParams& p);
// A call for which the layout kernel and a move of its own are faster than one launch (p.T, p.H, p.row_bytes, p.payload, the
// routing shape and the tile overrides set, p.fused = 1).
bool move_prefers_finished_layout(const MoveParams& p, int count_blocks);

// Column-major scales of an expanded dispatch on their way.  A row's scales belong into as many columns as it has scales, a
// dword each, 128 bytes of a column being the work of 32 rows that are moved far apart in time and by different XCDs: every
// such store is a partial line of its own.  So where the pad kernel follows, the move kernel stores a row's scales side by side
// and the pad kernel puts them into their columns.  Both in the same memory: the scales of 64 rows r0 .. r0 + 63 (the last
// block: what is left) occupy 64 dwords of every column, and in between these places hold the same block row by row.
constexpr int kScaleBlockRows = 64;
constexpr int kMaxBlockedScales = 128;     // scales of a row: the pad kernel turns a block in LDS

bool scales_in_blocks(const MoveParams& m, int alignment);

// What the move has left to do: blocked scales, and the padding rows if `rows`.
hipError_t launch_zero_padding(const PadParams& p, bool rows, hipStream_t stream);

// V1 (intranode) handle bookkeeping computed from is_token_in_rank, and the -1 fill of unused recv_topk_idx rows.
struct FillTailParams {
    int64_t* recv_topk_idx;          // [capacity, K]
    const int32_t* total_rows;       // device: rows in use
    int64_t capacity;
    int K;
};

hipError_t launch_fill_tail(const FillTailParams& p, hipStream_t stream);

// Rows of an expanded output that a call writes or zeroes, for the two sides of the memory-side cache: the dispatch and the combine of
// its rows have to come to the same answer, and these arguments are the same for both.  An output of exact size: all of it.  One of
// worst-case size (M tokens of each rank, M * min(K, E) + E * (alignment - 1) rows), with even routing: one alignment for each expert that
// has a row where next to none (two deviations) needs a second one, otherwise the selections and half an alignment for each.
inline double expanded_rows_in_use(int64_t rows, int64_t meta_rows, int T, int K, int E, int R, int M) {
    if (meta_rows < int64_t(M) * R) return double(rows);
    const double padding = std::max(double(rows) - double(M) * std::min(K, E), 0.0), alignment = padding / E + 1.0;
    const double selections = double(T) * K, each = selections / E;
    if (each + 2.0 * std::sqrt(each) <= alignment) return E * (1.0 - std::exp(-each)) * alignment;
    return selections + 0.5 * padding;
}
constexpr double kExpandedBytesInCache = 240e6;

struct CombineParams {
    const uint8_t* x;
    int64_t num_x_rows;
    const float* topk_weights;
    const uint8_t* bias0;
    const uint8_t* bias1;
    const int64_t* topk_idx;
    const int32_t* slot;
    const int32_t* meta;
    int64_t num_meta_rows;
    const int32_t* psum_rank;
    uint8_t* out;
    float* out_w;
    int T, H, K, E, R, E_l, rank_idx, M;
    int do_expand, multi_red;
    int tiles;
    int32_t* status;
    // V1 (intranode) conventions: slot is send_head [T, R] holding receive rows; terms are added in ascending
    // rank order; weights [rows, Kw] are summed over the token's rows.
    int rank_mode;
    int Kw;
    int vecs;            // forced column tile, 0 = choose
    int shares_tile;     // the rows are a BF16 dispatch's, on a finished layout (1) or in a single launch (2): kb_of_wavefront; 0: not, or not known
};

hipError_t launch_combine_kernel(CombineParams p, hipStream_t stream);
// KB of row a wavefront of it has.
int combine_tile(const CombineParams& p);

// dst_buffer_slot_idx of a handle rebuilt from its recv_src_metadata and per-rank prefix (see combine.hip).
struct SlotMapParams {
    const int32_t* meta;         // [num_meta_rows, K + 2]
    int64_t num_meta_rows;
    const int32_t* psum_rank;    // [R] inclusive
    int32_t* slot;               // [T, K] out
    int T, K, R, rank_idx, M;
};

hipError_t launch_rebuild_slot_map(const SlotMapParams& p, hipStream_t stream);

struct CastParams {
    const uint8_t* x;
    uint8_t* out;
    float* scales;
    int T, H;
};

hipError_t launch_cast_kernel(const CastParams& p, hipStream_t stream);

struct LLDispatchParams {
    int use_fp8;
    int round_scale, use_ue8m0;
    int S, src_rank_begin, src_token_stride;
    const int32_t* num_tokens_per_src;
    int H, K, E, expert_begin, E_l, R, M;
    const uint8_t* x;
    const int64_t* topk_idx;
    uint8_t* packed_x;
    float* packed_scales;
    int32_t* packed_count;
    int32_t* packed_src_info;
    int64_t* packed_layout_range;
    int32_t* cumulative_stats;
    int32_t* lane_slot;      // optional [S*stride, K]: packed row (le * rows + slot) of every (token, lane), -1 none
    // workspace
    int32_t* status;
    int32_t* chunk_counts;   // [E_l][C]: rows chunk c (256 tokens of one source) brings to a local expert
    int32_t* pos_expert;     // [S*stride*K]: position of a local selection inside its chunk
    // launch-shape overrides, 0 = choose
    int pairs, threads, two_kernels;
};

// Compute units of the current device (asked once per device).
int compute_units();

// Ranks a token's selections name, on average.  The rules of a call's launches ask for it several times over: with std::pow here
// choosing a small BF16 move took 0.65 us of the host, with a few products 0.39.
inline double distinct_ranks(int ranks, int selections) {
    double missed = 1.0;
    for (double factor = 1.0 - 1.0 / ranks; selections > 0; selections >>= 1, factor *= factor)
        if (selections & 1) missed *= factor;
    return ranks * (1.0 - missed);
}

// BF16 rows few enough to be read from the caches (T tokens that go to `rows` rows each): the KB of a row that a wavefront of the dispatch writes and
// a wavefront of the combine reads, the same for both, so that what an XCD has written it finds in its own L2 (0: each takes its own).
// Lines by wavefronts of 2 KB a CU.  Dispatch and combine, us, top-8 of 8 ranks unless said, rows combined as the dispatch has left them / with a pass
// in between that reads them and writes as many others, which are combined:
//   two launches                    1 KB both     2 KB both      4 and 1 KB (2 and 1 KB)
//     128 x 1024 top-2 of 2   1     10.5 / 12.7   10.9 / 13.0    10.9 / 12.9      up to 4: 1 KB, which has twice the wavefronts
//     256 x 1024              1     12.9 / 16.8   13.5 / 17.4    14.5 / 17.3
//     146 x 7168              4     14.5 / 26.9   14.5 / 26.8    18.4 / 26.9
//     292 x 7168              8     18.4 / 29.9   18.1 / 30.1    25.5 / 30.4      up to 30: 2 KB
//     1706 x 2888             20    35.8 / 53.0   32.4 / 50.3    35.5 / 49.5
//     950 x 7168              26    40.6 / 63.0   39.1 / 60.7    41.6 / 60.4
//     1243 x 7168             34    49.8 / 78.2   47.9 / 76.9    49.0 / 74.8      left alone (2901 x 2888 50.6 / 76.8, 48.7 / 74.8, 48.0 / 71.9)
//     512 x 7168 expanded     14    34.2 / 52.0   34.6 / 53.0    37.4 / 51.2      tokens of seven and a half rows and more: 1 KB up to 15
//     320 x 8192              5     15.6 / 23.9   16.1 / 27.8    22.5 / 26.2      rows of whole 8 KB (256 x 4096 top-4 12.3 / 18.9, 12.5 / 20.5): 1 KB up to 6
//   a single launch
//     73 x 7168               2     15.2 / 21.6   14.1 / 20.6    15.9 / 20.5      up to 22: 2 KB
//     292 x 7168 of 32        8     20.5 / 33.4   19.6 / 32.4    26.9 / 34.0
//     731 x 7168              20    32.1 / 49.5   29.4 / 46.9    32.2 / 46.6
//     950 x 7168              26    40.6 / 62.2   44.4 / 67.5    37.6 / 56.9      left alone
//     320 x 4096              5     17.4 / 26.6   18.5 / 28.9    21.1 / 27.3      rows of whole 8 KB: 1 KB from 4 to 6 (155 x 4096, one row, 2.4 a CU 17.7, 17.1)
//     146 x 7168 expanded     4     20.8 / 32.1   21.4 / 33.2    25.8 / 32.5      tokens of seven and a half rows and more: 1 KB up to 4
// Rows that leave a fourth of their 2 KB tiles empty take 1 KB (2362 x 1064 23.9 / 38.4, with 2 KB 24.7 / 39.2), in a single launch only tokens of many.
// Past the lines of a single launch its combine has the tile of two launches, which a cached dispatch on the same handle has (shared_tile); behind the single
// launch that is level with its own (950 x 7168 37.7 / 56.8 with 2 KB, 37.6 / 56.9 with 1 KB).  A combine whose rows are not those of a BF16 dispatch keeps to its own rule
// below 18 a CU: fused cast, 1 / 2 KB, 1194 x 2944 21.4 / 22.0, 3584 x 1024 22.4 / 22.9, 192 x 4096 19.9 / 21.1; 1706 x 2944 top-4 22.2 / 21.3, 731 x 7168 25.6 / 25.8.
// V1 handles do not say what made them, and the combine behind FP8 rows is ahead with 1 KB up to 8 a CU, BF16 level or ahead there: FP8, 1 / 2 KB, 200 x 7168 18.0 / 18.6, 400 x 4096
// 19.3 / 20.0, 560 x 2048 19.6 / 19.9, 290 x 7168 20.4 / 20.8;  BF16 19.5 / 19.9, 20.3 / 21.0, 20.8 / 20.8, 21.8 / 21.9.  Level from 8 on (FP8, 682 x 2944 34.2 / 34.3, 512 x 4096 33.2 / 33.9).
inline int kb_of_wavefront(int64_t T, int row_bytes, double rows, bool single_launch, bool v1) {
    const int kb = (row_bytes + 1023) / 1024, tiles = (kb + 1) / 2;
    const int64_t cus = compute_units(), wavefronts = T * tiles;
    if (row_bytes < tiles * 1536) return T * kb <= cus * (single_launch ? 12 : 30) && (rows >= 6.5 || !single_launch) ? 1 : 0;
    if (wavefronts > cus * (single_launch ? 22 : 30)) return 0;
    const bool many = rows >= 7.5, whole_8kb = row_bytes % 8192 == 0;
    if (single_launch && whole_8kb && !many) return wavefronts > cus * 4 && wavefronts <= cus * 6 ? 1 : 2;
    const int one_kb_to = single_launch ? (whole_8kb ? 6 : many ? 4 : 0) : many ? 15 : v1 ? 8 : whole_8kb ? 6 : 4;
    return wavefronts <= cus * one_kb_to ? 1 : 2;
}

// The tile of the combine, and of a dispatch on the handle, where the handle is a single launch's or not.
inline int shared_tile(int64_t T, int row_bytes, double rows, bool single_launch, bool v1) {
    const int kb = single_launch ? kb_of_wavefront(T, row_bytes, rows, true, v1) : 0;
    return kb != 0 ? kb : kb_of_wavefront(T, row_bytes, rows, false, v1);
}

// LDS a workgroup asks for so that a CU holds at most `per_cu` of them (0: no limit).
size_t lds_for_residency(int per_cu);

// Threads of a workgroup where the dispatch is a single kernel, 0 where it is the counting and the move kernel.
int ll_single_kernel_threads(const LLDispatchParams& p);
hipError_t launch_ll_dispatch(const LLDispatchParams& p, hipStream_t stream);

struct LLCombineParams {
    int S, src_rank_begin, src_token_stride;
    const int32_t* num_tokens_per_src;
    int H, K, E, expert_begin, E_l, R, M;
    const uint8_t* x;
    const int64_t* topk_idx;
    const float* topk_weights;
    const int32_t* src_info;
    const int64_t* layout_range;
    const int32_t* lane_slot;    // optional: what the dispatch recorded; replaces the search through src_info
    uint8_t* out;
    int32_t* status;
    int vecs;                    // forced column tile, 0 = choose
    int use_logfmt;              // gathered rows pass through the LogFMT-10 codec
};

hipError_t launch_ll_combine(const LLCombineParams& p, hipStream_t stream);

}  // namespace deep_ep_hip
