// Combine for gfx950: per origin token, gather the rows that came back, accumulate in fp32 in a
// fixed order on top of the optional biases, round once to BF16 and store.
//
// Replaces deep_ep/include/deep_ep/impls/combine.cuh:86-237 (send side, optional local reduce of
// expanded rows) and deep_ep/include/deep_ep/impls/combine_reduce_epilogue.cuh:62-142 with
// combine_utils.cuh:111-168 (ordered fp32 reduce): on one GPU the returned rows already sit in
// local HBM, so the two kernels become one gather-reduce indexed by the dispatch handle.
//
// Order of accumulation (fixed, so results are reproducible): bias_0 + bias_1 first, then one
// term per distinct destination rank in ascending order of that rank's master (highest) lane.
// Expanded layout with multiple reduction: each rank's term is the fp32 sum of that rank's rows in
// lane order rounded to BF16.  Expanded layout without multiple reduction: every valid lane is its
// own term, in lane order.
//
// One wavefront owns one (token, column tile of kVecs * 512 channels).  Large calls are bound by memory, small ones by the chain
// of trips to it: routing loads, rows of the first batch, rows of the second.  With a start that waited for the index, biases and
// weights waited for in front of the rows and a branch around every load it took (combine kernel and its launch, us before ->
// now): 1237 x 2888 top-9 over 6 ranks 11.5 -> 9.8, 4096 x 2048 top-6 19.1 -> 17.3, 8192 x 7168 4 of 4 ranks 73.9 -> 67.6,
// 8192 x 7168 top-8 over 8 ranks 118.4 -> 117.0 and 16384 over 32 ranks 333 -> 321 (1.9 GB, 5.8 TB/s -> 6.0).  Eight rows
// a batch instead of four measured the same.
#include <algorithm>
#include <cmath>

#include "device_utils.h"
#include "kernels.h"
#include "../../include/deep_ep_hip.h"

namespace deep_ep_hip {

namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWaveSize;
#ifndef DEEP_EP_HIP_COMBINE_BATCH
#define DEEP_EP_HIP_COMBINE_BATCH 4
#endif
constexpr int kBatch = DEEP_EP_HIP_COMBINE_BATCH;   // source rows whose loads are issued together

template <int kVecs>
__device__ __forceinline__ void add_row(float (&acc)[kVecs][8], const vec16 (&v)[kVecs]) {
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
        acc[i][0] += bf16_lo(v[i].x); acc[i][1] += bf16_hi(v[i].x);
        acc[i][2] += bf16_lo(v[i].y); acc[i][3] += bf16_hi(v[i].y);
        acc[i][4] += bf16_lo(v[i].z); acc[i][5] += bf16_hi(v[i].z);
        acc[i][6] += bf16_lo(v[i].w); acc[i][7] += bf16_hi(v[i].w);
    }
}

// The row is the same for the whole wavefront, so it is read through a buffer descriptor of its own (base: the row; range:
// its bytes, none for row < 0): channels past the row's end and missing rows read as zero in the load itself.  With a branch
// around each load instead, the compiler put waits and address arithmetic between the loads of a batch.
template <int kVecs, bool kStream>
__device__ __forceinline__ void load_row(vec16 (&v)[kVecs], const uint8_t* base, int row, int row_bytes, int tile, int lane) {
    const auto of_row = buffer_of(base + int64_t(max(row, 0)) * row_bytes, row >= 0 ? row_bytes : 0);
#pragma unroll
    for (int i = 0; i < kVecs; ++i) v[i] = buffer_load16_as<kStream>(of_row, (tile * kVecs + i) * 1024 + lane * 16);
}

// acc += sum of rows named by the lanes in `mask` (ascending lane order); row_of_lane < 0 adds nothing.
template <int kVecs, bool kStream>
__device__ __forceinline__ void accumulate_rows(float (&acc)[kVecs][8], uint64_t mask, int row_of_lane,
                                                const uint8_t* x, int row_bytes, int tile, int lane) {
    while (mask) {
        int rows[kBatch];
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            rows[b] = -1;
            if (mask) {
                const int j = __builtin_ctzll(mask);
                mask &= mask - 1;
                rows[b] = read_lane(row_of_lane, j);
            }
        }
        vec16 v[kBatch][kVecs];
#pragma unroll
        for (int b = 0; b < kBatch; ++b) load_row<kVecs, kStream>(v[b], x, rows[b], row_bytes, tile, lane);
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
            if (rows[b] >= 0) add_row<kVecs>(acc, v[b]);
    }
}

// kLayout: what the rows of x are.  Each gets a kernel of its own, so that the sequencing registers of the expanded
// layout do not cost the compact layout occupancy.
// kRankRows: V1 conventions (CombineParams::rank_mode).
enum : int { kCompactRows = 0, kExpandedRows = 1, kExpandedRowsReducedPerRank = 2, kRankRows = 3 };

// kStream: rows are read past the memory-side cache (reads_past_the_cache).
template <int kVecs, int kLayout, bool kStream>
__global__ __launch_bounds__(kThreads) void combine_kernel(const CombineParams p) {
    constexpr bool kExpanded = kLayout == kExpandedRows || kLayout == kExpandedRowsReducedPerRank;
    const int lane = threadIdx.x & 63;
    const unsigned work = wave_work_index(blockIdx.x, kWavesPerBlock);
    if (work >= unsigned(p.T) * unsigned(p.tiles)) return;
    const int t = int(work / unsigned(p.tiles));
    const int tile = int(work - unsigned(t) * unsigned(p.tiles));
    const int row_bytes = p.H * 2;

    // Routing of this token: lanes [0, K).  Indices, slots and the ends of the ranks' regions (lane r: rank r) are asked for
    // together, on clamped columns instead of behind branches, and the biases with them: where a rank's region starts then
    // comes from another lane, not from a load that waits for the index.
    const int64_t at = int64_t(t) * p.K + min(lane, p.K - 1);
    const int slot = p.slot[at];
    int64_t raw = -1;
    int rank_end = 0;
    if constexpr (kLayout != kRankRows) {
        raw = p.topk_idx[at];
        rank_end = p.psum_rank[min(lane, p.R - 1)];
    }

    float acc[kVecs][8];
#pragma unroll
    for (int i = 0; i < kVecs; ++i)
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[i][c] = 0.f;
    if (p.bias0 != nullptr) {
        vec16 v[kVecs];
        load_row<kVecs, true>(v, p.bias0, t, row_bytes, tile, lane);
        add_row<kVecs>(acc, v);
    }
    if (p.bias1 != nullptr) {
        vec16 v[kVecs];
        load_row<kVecs, true>(v, p.bias1, t, row_bytes, tile, lane);
        add_row<kVecs>(acc, v);
    }

    int e = -1, d = -1, row_c = -1, my_row = -1, erow = -1;
    if constexpr (kLayout == kRankRows) {
        // V1 handle: lane q < R reads the receive row of this token on rank q; rows are added in ascending
        // rank order and the weights of all rows are summed (csrc/kernels/legacy/intranode.cu:940-1033).
        if (lane < p.K && slot >= 0) {
            if (slot < p.num_x_rows) row_c = slot;
            else atomicOr(p.status, DEEP_EP_HIP_STATUS_ROW_OVERFLOW);
        }
        uint64_t rows = __ballot(row_c >= 0);
        if (tile == 0 && p.out_w != nullptr) {
            float w = 0.f;
            while (rows) {                                        // by all lanes: any of them is read from
                const int j = __builtin_ctzll(rows);
                rows &= rows - 1;
                const int row = read_lane(row_c, j);
                if (p.topk_weights != nullptr && lane < p.Kw) w += p.topk_weights[int64_t(row) * p.Kw + lane];
            }
            if (lane < p.Kw) p.out_w[int64_t(t) * p.Kw + lane] = w;
        }
    } else {
        if (lane < p.K && raw >= 0 && raw < p.E) {
            e = int(raw);
            d = small_div(e, 1.0f / float(p.E_l));
        }
        int start = __shfl(rank_end, max(d - 1, 0) & 63, kWaveSize);
        if (p.R > kWaveSize && d > 0) start = p.psum_rank[d - 1];
        if (e >= 0 && slot >= 0) {
            row_c = (d > 0 ? start : 0) + (slot - p.rank_idx * p.M);
            if (!kExpanded && row_c >= p.num_x_rows) {
                atomicOr(p.status, DEEP_EP_HIP_STATUS_ROW_OVERFLOW);
                row_c = -1;
            }
        }
    }
    const bool returns_weights = kLayout != kRankRows && tile == 0 && p.out_w != nullptr;
    if (kExpanded || returns_weights) {
        for (int j = 0; j < p.K; ++j) {
            const int dj = read_lane(d, j);
            const int rj = read_lane(row_c, j);
            if (d >= 0 && dj == d && rj >= 0) my_row = rj;
        }
    }
    if (kExpanded && my_row >= 0 && my_row < p.num_meta_rows) {
        erow = p.meta[int64_t(my_row) * (p.K + 2) + 2 + lane];
        if (erow >= p.num_x_rows) {
            atomicOr(p.status, DEEP_EP_HIP_STATUS_ROW_OVERFLOW);
            erow = -1;
        }
    }

    // Weights travel back to the lane that owns them: asked for in front of the rows, stored behind them, so that the rows
    // are not held up by the wait.
    float w = 0.f;
    if (returns_weights && p.topk_weights != nullptr && lane < p.K) {
        if (kExpanded) {
            if (erow >= 0) w = p.topk_weights[erow];
        } else if (my_row >= 0) {
            w = p.topk_weights[int64_t(my_row) * p.K + lane];
        }
    }

    if constexpr (kLayout == kCompactRows || kLayout == kRankRows) {
        accumulate_rows<kVecs, kStream>(acc, __ballot(row_c >= 0), row_c, p.x, row_bytes, tile, lane);
    } else if constexpr (kLayout == kExpandedRows) {
        accumulate_rows<kVecs, kStream>(acc, __ballot(erow >= 0), erow, p.x, row_bytes, tile, lane);
    } else {
        // One term per destination rank, in ascending order of the rank's master lane; a rank's rows are summed in
        // lane order and the sum is rounded to BF16 before it is added.  The rows are put into that order first (each
        // lane learns the place of its row in the sequence), so that their loads go out kBatch at a time across the
        // ranks: a load round per rank would cost a memory round trip for one or two rows each.
        int place = -1, ends_term = 0, alone = 0, total = 0;
        uint64_t masters = __ballot(row_c >= 0);
        while (masters) {
            const int j = __builtin_ctzll(masters);
            masters &= masters - 1;
            const int dj = read_lane(d, j);
            const uint64_t members = __ballot(d == dj && erow >= 0);
            if (d == dj && erow >= 0) {
                place = total + __popcll(members & ((uint64_t(1) << lane) - 1));
                ends_term = (members >> lane) == 1 ? 1 : 0;
                alone = __popcll(members) == 1 ? 1 : 0;         // its BF16 round trip is exact: added as it is
            }
            total += __popcll(members);
        }
        const int flags_of_lane = ends_term | (alone << 1);
        float part[kVecs][8];
#pragma unroll
        for (int i = 0; i < kVecs; ++i)
#pragma unroll
            for (int c = 0; c < 8; ++c) part[i][c] = 0.f;
        for (int first = 0; first < total; first += kBatch) {
            int rows[kBatch], flags[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                rows[b] = -1;
                flags[b] = 0;
                if (first + b < total) {
                    const int j = __builtin_ctzll(__ballot(place == first + b));
                    rows[b] = read_lane(erow, j);
                    flags[b] = read_lane(flags_of_lane, j);
                }
            }
            vec16 v[kBatch][kVecs];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) load_row<kVecs, kStream>(v[b], p.x, rows[b], row_bytes, tile, lane);
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                if (rows[b] < 0) continue;
                if (flags[b] & 2) {
                    add_row<kVecs>(acc, v[b]);
                    continue;
                }
                add_row<kVecs>(part, v[b]);
                if (flags[b] & 1) {
#pragma unroll
                    for (int i = 0; i < kVecs; ++i)
#pragma unroll
                        for (int c = 0; c < 8; ++c) {
                            acc[i][c] += __uint_as_float(f32_to_bf16_bits(part[i][c]) << 16);
                            part[i][c] = 0.f;
                        }
                }
            }
        }
    }

    uint8_t* dst = p.out + int64_t(t) * row_bytes;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
        const int off = (tile * kVecs + i) * 1024 + lane * 16;
        if (off < row_bytes) {
            vec16 o;
            o.x = pack_bf16x2(acc[i][0], acc[i][1]);
            o.y = pack_bf16x2(acc[i][2], acc[i][3]);
            o.z = pack_bf16x2(acc[i][4], acc[i][5]);
            o.w = pack_bf16x2(acc[i][6], acc[i][7]);
            store16_stream(dst + off, o);
        }
    }
    if (returns_weights && lane < p.K) p.out_w[int64_t(t) * p.K + lane] = w;
}

// Rows a token has, on average: as if its experts were chosen evenly, and no more than there are.
double rows_per_token(const CombineParams& p) {
    const double returned = double(p.num_x_rows) / p.T;
    const int selections = p.rank_mode ? p.Kw : p.K;
    if (selections == 0) return returned;
    const int ranks = p.rank_mode ? p.K : p.R;
    return std::min(returned, p.do_expand && !p.rank_mode ? double(selections) : distinct_ranks(ranks, selections));
}

// How many workgroups a CU should hold at a time (0: the eight its registers allow).  Scattered rows stream fastest when not
// too many are under way.  us with 8 / 6 / 5 / 4 per CU, 1 KB tiles, top-8, hidden 7168 unless said:
//   8 ranks (5.3 rows a token)   4096 tokens  60.0 / 59.5 / 60.3 / 63.2;   8192  119.6 / 117.0 / 117.5 / 123.7;  16384  247 / 237 / 233 / 247
//   16 ranks (6.4)               8192 tokens 149.1 / 145.4 / 141.7 / 143.8;  16384  303 / 297 / 287 / 286
//   32 ranks (7.2)               4096 tokens  81.3 / 80.1 / 78.5 / 78.6;   16384  336 / 330 / 321 / 312
//   4 of 4 ranks (2.7)           8192 tokens  67.6 / 71.3 / 76.0;   16384 x 2048 top-6 (4.4) 60.9 / 62.2 / 64.1
//   top-6 of 8 ranks (4.4)       4096 tokens  53.5 / 52.6 / 54.0;   8192  103.4 / 100.6 / 102.8;   16384  210 / 199 / 202
//   top-4 of 16 ranks (3.6)      8192 tokens  88.1 / 87.3 / 88.7;   16384  176 / 172 / 175;   of 8 ranks (3.3)   158 / 157 / 162
//   2048 channels (32768 tokens) 8 ranks 142 / 139 / 139;                64 ranks 205 / 199 / 195
//   8192 channels (16384 tokens) top-6 of 8 ranks 238 / 247 / 252;   4096 channels (8192) of 64 ranks 79.5 / 83.2 / 83.2: rows a
//   power of two apart are left alone
//   a GB of rows and seven a token, of whole KB, a dispatch in front, 6 / 5 / 4: 16384 x 7168 of 32 ranks 669.8 / 659.2 / 653.6, of 64 713 / 705.6 /
//   697.4;   16000 x 6144 565 / 558.3 / 554.3;   20000 x 5120 587 / 578.2 / 576.8;   behind a fused cast, 16384 x 7168 of 32 541.7 / 538.2 / 527.9;   other
//   rows 12000 x 6000 of 32 455.2 / 454.0 / 456.4;   14000 x 7000 of 64 681.9 / 676.2 / 676.4
//   whole passes with 5 / 4: 6000 x 7168 of 32 (619 MB) 252.8 / 254.8; V1 12000 x 5120 of 32 372.4 / 383.9; 30000 x 3072 of 32 547.1 / 549.9; 16384 x 7168 of 64, cast, 615.6 / 604.3
//   from 500 MB on: 8000 x 5120 of 16 (532 MB) 188.2 without, 184.2 with five; 10000 x 5000 of 8 (530 MB) 241.6, 239.4 with six; 8307 x 4736 of 32 ranks behind a cast (567 MB) 181.7 without a limit, 178.6 with five
// Smaller calls lose by any limit (4096 x 2048 top-6: 17.3 / 18.3), and so do narrower rows (65536 x 768 over 16 ranks 125 / 137 /
// 146).
// The limit is kept with LDS, which a product on another stream then lacks: beside products of 4096^3 BF16 that share the GPU,
// twenty combines and 24 products together take 4.44 ms without it and 4.58 with six at 8192 tokens over 8 ranks (alone 122 and
// 119 us a combine), 8.24 and 8.45 with five at 16384 over 32 (337 and 322).  Expanded rows are left alone: there it gave 1 %
// alone (187.7 and 185.6) and took 4 % beside products (5.68 and 5.93).
int workgroups_per_cu(const CombineParams& p) {
    const double rows = rows_per_token(p), bytes = rows * p.T * p.H * 2;
    if ((p.do_expand && !p.rank_mode) || p.H < 2048 || p.H % 4096 == 0) return 0;
    if (p.H < 6144 ? rows < 5.0 || bytes < 500e6 : rows >= 5.0 ? bytes < 300e6 : rows < 3.5 || bytes < 450e6) return 0;
    if (rows >= 7.0 && bytes >= 1e9 && p.H >= 5120 && p.H % 512 == 0 && !p.rank_mode) return 4;
    return rows >= 5.8 ? 5 : 6;
}

// The rows a combine adds up have just been written, by the experts or by the dispatch itself: up to 110 MB of them are read with plain
// loads, which find them in the memory-side cache.  Dispatch and combine of BF16 rows, us, streaming / plain rows (the dispatch stores
// by the same line, for the rows even routing would give, cached_side): 4096 x 2048 top-6 of 8 ranks, forward and backward (74 MB) 91.2 / 84.9, 16384 x 2048 of 2 ranks (100 MB) 77.5
// / 76.0; combine of rows an expert has just written, with an FP8 dispatch in front, 1024 x 7168 (78 MB) 42.3 / 36.7, 700 x 4096 (30 MB) 27.4 /
// 26.6; rows that are in HBM while the cache is full of what others have written are the other way round (41.0 / 53.5).  More rows than
// the cache holds beside other traffic are read past it: 2100 x 7168 (160 MB) 67.5 / 74.0, 4096 x 7168 (311 MB) 134 / 170.  So are
// expanded rows among padding rows that are zeroed behind them, from 240 MB of both on: top-8, aligned to 128, input just written, 400 x 7168 of
// 128 experts (46 of 235 MB) 16.3 / 15.1, of 144 (264 MB) 16.3 / 16.2, of 160 (294 MB) 16.7 / 23.7, 300 x 7168 of 256 (470 MB) 14.9 / 23.8.
bool reads_past_the_cache(const CombineParams& p) {
    const double row_bytes = p.H * 2.0;
    const bool between_padding = p.do_expand && !p.rank_mode && expanded_rows_in_use(p.num_x_rows, p.num_meta_rows, p.T, p.K, p.E, p.R, p.M) * row_bytes > kExpandedBytesInCache;
    return between_padding || rows_per_token(p) * p.T * row_bytes > 110e6;
}

// Column tile per wavefront: 1 KB of a BF16 row (512 channels, 41 registers, eight wavefronts per SIMD), or 2 KB, which repeats the routing
// work half as often and has half the wavefronts to hide its loads with.  2 KB for few rows a token (top-2, or two ranks), where the routing is
// as much as the rows, from three quarters of the places on, where kb_of_wavefront does not settle it; V1 rows, whose routing is shorter, from a full round on.  Change by 2 KB tiles in %
// at 0.55 / 0.8 / 1.0 / 1.1 / 1.4 / 4 times as many wavefronts of 1 KB as places (730 shapes, rows of 2 to 14 KB):
//   compact, top-2 of 2 ranks, 8 KB rows    +1.2 / -2.2 / -4.0 / -8.0 / -7.6 / -8.5;   top-2 of 8 ranks +0.6 / +0.5 / -1.5 / -5.8 / -8.2 / -4.4
//   expanded, top-2                          +0.5 / -3.0 / -6.1 / -7.9 / -1.3 / -2.7
//   V1, top-2 of 8 ranks, 4 KB rows          +2.4 / +3.2 / +1.0 / -5.8 / -5.1
//   more rows a token, up to one round: compact top-8 of 8 ranks -3 to +5, expanded top-8 -2 to +9, V1 top-8 -1 to +9
// A last tile that is half idle costs what the others gain: rows of 3 KB, expanded, top-2, 0.0 / +3.0 / +12.3 / +4.6 / +1.6 / +5.4; compact
// +0.6 / -0.5 / +2.0 / -7.1 / -8.1 / -2.2.
bool takes_two_kb_tiles(const CombineParams& p) {
    const int kb = (p.H * 2 + 1023) / 1024;
    if (!reads_past_the_cache(p)) {
        const int same = shared_tile(p.T, p.H * 2, rows_per_token(p), p.shares_tile == 2, p.rank_mode != 0);
        const bool others = p.shares_tile == 0 && int64_t(p.T) * ((kb + 1) / 2) < int64_t(compute_units()) * 18;
        if (same != 0 && !others) return same == 2;
    }
    if (kb < 2 || rows_per_token(p) >= 2.3) return false;
    const int64_t places = int64_t(compute_units()) * 8 * kWavesPerBlock, waves = int64_t(p.T) * kb;
    if (p.rank_mode) return waves > places;
    const bool half_idle = kb % 2 == 1 && kb < 8;
    return 4 * waves >= 3 * places && (!half_idle || (!p.do_expand && waves > places));
}

template <int kVecs, int kLayout>
hipError_t launch_layout(const CombineParams& p, unsigned blocks, hipStream_t stream) {
    const auto kernel = reads_past_the_cache(p) ? combine_kernel<kVecs, kLayout, true> : combine_kernel<kVecs, kLayout, false>;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), lds_for_residency(workgroups_per_cu(p)), stream, p);
    return hipGetLastError();
}

template <int kVecs>
hipError_t launch(CombineParams p, hipStream_t stream) {
    const int row_bytes = p.H * 2;
    p.tiles = (row_bytes + kVecs * 1024 - 1) / (kVecs * 1024);
    const int64_t waves = int64_t(p.T) * p.tiles;
    const unsigned blocks = unsigned((waves + kWavesPerBlock - 1) / kWavesPerBlock);
    if (p.rank_mode) return launch_layout<kVecs, kRankRows>(p, blocks, stream);
    if (!p.do_expand) return launch_layout<kVecs, kCompactRows>(p, blocks, stream);
    if (!p.multi_red) return launch_layout<kVecs, kExpandedRows>(p, blocks, stream);
    return launch_layout<kVecs, kExpandedRowsReducedPerRank>(p, blocks, stream);
}

// ---- the token -> received-row map of a handle, rebuilt from the rows' own records ----
// A compact receive row r carries (source rank * M + token, source rank * K + master lane) in the first two columns of
// recv_src_metadata, and the rows of destination rank d are [psum[d - 1], psum[d]): so row r is slot r - psum[d - 1] of
// the master lane of its token.  Every other entry is -1.
__global__ __launch_bounds__(kThreads) void fill_slot_map_kernel(int32_t* slot, int64_t n) {
    for (int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x; i < n; i += int64_t(gridDim.x) * kThreads) slot[i] = -1;
}

__global__ __launch_bounds__(kThreads) void scatter_slot_map_kernel(const SlotMapParams p) {
    extern __shared__ int32_t psum[];      // [R]
    for (int i = threadIdx.x; i < p.R; i += kThreads) psum[i] = p.psum_rank[i];
    __syncthreads();
    const int64_t rows = min(int64_t(psum[p.R - 1]), p.num_meta_rows);
    for (int64_t r = int64_t(blockIdx.x) * kThreads + threadIdx.x; r < rows; r += int64_t(gridDim.x) * kThreads) {
        const int token = p.meta[r * (p.K + 2)] - p.rank_idx * p.M;
        const int lane = p.meta[r * (p.K + 2) + 1] - p.rank_idx * p.K;
        if (token < 0 || token >= p.T || lane < 0 || lane >= p.K) continue;       // a row of another source rank
        int lo = 0, hi = p.R - 1;                 // first d with r < psum[d]
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (r < psum[mid]) hi = mid;
            else lo = mid + 1;
        }
        const int first = lo > 0 ? psum[lo - 1] : 0;
        p.slot[int64_t(token) * p.K + lane] = p.rank_idx * p.M + int(r - first);
    }
}

}  // namespace

hipError_t launch_rebuild_slot_map(const SlotMapParams& p, hipStream_t stream) {
    const int64_t n = int64_t(p.T) * p.K;
    if (n == 0) return hipSuccess;
    const unsigned fill_blocks = unsigned(std::min<int64_t>((n + kThreads - 1) / kThreads, 2048));
    hipLaunchKernelGGL(fill_slot_map_kernel, dim3(fill_blocks), dim3(kThreads), 0, stream, p.slot, n);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess || p.num_meta_rows == 0) return err;
    const unsigned blocks = unsigned(std::min<int64_t>((p.num_meta_rows + kThreads - 1) / kThreads, 2048));
    hipLaunchKernelGGL(scatter_slot_map_kernel, dim3(blocks), dim3(kThreads), size_t(p.R) * sizeof(int32_t), stream, p);
    return hipGetLastError();
}

int combine_tile(const CombineParams& p) {
    if (p.vecs != 0) return p.vecs == 1 || p.vecs == 4 ? p.vecs : 2;
    return p.T > 0 && takes_two_kb_tiles(p) ? 2 : 1;
}

hipError_t launch_combine_kernel(CombineParams p, hipStream_t stream) {
    if (p.T == 0) return hipSuccess;
    switch (combine_tile(p)) {
        case 1: return launch<1>(p, stream);
        case 4: return launch<4>(p, stream);
        default: return launch<2>(p, stream);
    }
}

}  // namespace deep_ep_hip
