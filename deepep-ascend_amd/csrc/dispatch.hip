// Dispatch payload movement for gfx950: every token row is read once from HBM and written once per
// destination row (compact: one row per distinct destination rank; expanded: one row per valid
// (token, lane)), with the optional BF16 -> FP8 e4m3 per-1x128 cast fused between the load and
// the stores.
//
// Replaces the per-token warp loop of deep_ep/include/deep_ep/impls/dispatch.cuh:259-395 together
// with the receive-side copy of deep_ep/include/deep_ep/impls/dispatch_copy_epilogue.cuh:70-208:
// on one GPU the "send buffer -> peer recv buffer -> output tensor" chain collapses into a single
// scatter.  Slot numbers come from the layout pass (scan based, deterministic) instead of atomics.
//
// Work decomposition: one wavefront owns one (token, column tile).  All 16-byte loads of the tile
// are issued first, then the routing metadata is resolved while they are in flight, then the tile
// is stored to each destination with 16-byte stores.
//
// Single-launch mode ("fused"): the first workgroups of the grid are counting workgroups (one 256-token
// chunk each, the code of the layout kernel) and one publishing workgroup that writes the handle tensors.
// Mover workgroups issue their payload loads, then read the chunk totals and position words the counting
// workgroups store (again, until a word shows the tag of this launch), and work their row numbers out from
// those.  Counting workgroups have the lowest workgroup ids, wait for nothing and are therefore resident
// before any mover can wait for them; every wait is bounded.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "device_utils.h"
#include "fp8_cast.h"
#include "kernels.h"
#include "layout_count.h"
#include "publish.h"
#include "../../include/deep_ep_hip.h"

namespace deep_ep_hip {

namespace {

#ifndef DEEP_EP_HIP_MOVE_THREADS
#define DEEP_EP_HIP_MOVE_THREADS 256
#endif
constexpr int kThreads = DEEP_EP_HIP_MOVE_THREADS;
constexpr int kWavesPerBlock = kThreads / kWaveSize;

// Per-lane routing state of one token, lanes [0, K) meaningful.
struct Route {
    int e;        // expert id or -1
    int d;        // destination rank or -1
    int row_c;    // compact row, on master lanes only (else -1)
    int my_row;   // compact row of this lane's destination (all valid lanes)
    int erow;     // expanded row (expanded layout), else -1
    float w;
};

// A word of the layout tables a finished layout pass (an earlier launch, or a cached handle) left in memory.
__device__ __forceinline__ int layout_word(const int32_t* at) {
    return *at;
}

// What the caller gave for one (token, lane): independent of the layout pass, so a single-launch dispatch loads
// it together with the payload, before it knows that the layout is complete.
struct RouteInputs {
    int64_t raw;         // topk_idx entry
    uint8_t mask_byte;   // is_token_in_rank entry (mask routing)
    float w;             // topk_weights entry
};

__device__ __forceinline__ RouteInputs load_route_inputs(const MoveParams& p, int t, int lane) {
    RouteInputs in{-1, 0, 0.f};
    if (lane < p.K) {
        const int64_t at = int64_t(t) * p.K + lane;
        if (p.route_mask != nullptr) in.mask_byte = p.route_mask[at];
        else if (!(p.cached && p.rank_lanes)) in.raw = p.topk_idx[at];
        if (p.topk_weights != nullptr) in.w = p.topk_weights[at];
    }
    return in;
}

// The word of the layout pass for (token, lane): the cached handle's slot, or the position word (kernels.h).
__device__ __forceinline__ uint32_t load_position_word(const MoveParams& p, int t, int lane) {
    if (lane >= p.K) return 0xffffffffu;
    const int32_t* words = p.cached ? p.cached_slot : reinterpret_cast<const int32_t*>(p.pos);
    return uint32_t(layout_word(words + int64_t(t) * p.K + lane));
}

// Single-launch dispatch: flat_bases is this workgroup's LDS copy of the exclusive prefix over the chunk totals of the
// rank buckets, expert_base the first expanded row of (the token's chunk, the lane's expert).
template <bool kFused>
__device__ __forceinline__ Route resolve_route(const MoveParams& p, const RouteInputs& in, uint32_t word, const int* flat_bases,
                                               int expert_base, int t, int lane, bool first_tile) {
    Route r{-1, -1, -1, -1, -1, in.w};
    const int chunk = t / kLayoutChunk;

    // ---- issue every load that does not depend on another one, then consume: one memory round trip ----
    int64_t raw = in.raw;
    const uint8_t mask_byte = in.mask_byte;
    const bool rank_lanes_cached = p.cached && p.rank_lanes;
    // Wave lane q < R fetches the base row of (rank q, this token's chunk) and the start of rank q's bucket; the
    // routing lanes pick theirs up by shuffle.  (More than 64 ranks: each master lane fetches its own pair below.)
    const bool bases_by_lane = !kFused && !p.cached && p.R <= kWaveSize;
    int base_of_rank = 0, start_of_rank = 0;
    if (bases_by_lane && lane < p.R) {
        base_of_rank = layout_word(p.tab.rank_bases + int64_t(lane) * p.tab.chunks_padded + chunk);
        start_of_rank = layout_word(p.tab.rank_bases + int64_t(lane) * p.tab.chunks_padded);
    }

    int slot = -1, epos = -1;
    const int cached_v = int(word);
    const uint32_t packed = word;
    if (lane < p.K) {
        if (rank_lanes_cached) {
            // V1 cached dispatch: send_head names the receive row of every (token, rank) pair
            if (cached_v >= 0) r.e = lane;
            slot = cached_v;
        } else {
            if (p.route_mask != nullptr) raw = mask_byte != 0 ? int64_t(lane) : int64_t(-1);
            if (raw >= 0 && raw < p.E) r.e = int(raw);
            if (p.cached) {
                slot = cached_v >= 0 ? cached_v - p.rank_idx * p.M : -1;
            } else {
                slot = (packed & kNoPosition) == kNoPosition ? -1 : int(packed & kNoPosition);
                epos = int((packed >> kExpertPositionShift) & kNoPosition);
            }
        }
    }
    if (r.e >= 0) r.d = small_div(r.e, p.rcp_E_l);
    else slot = -1;
    if (!p.cached) {
        int base, start;
        if constexpr (kFused) {
            const int row = (r.d >= 0 && slot >= 0 ? r.d : 0) * p.tab.chunks_padded;
            base = flat_bases[row + chunk];
            start = flat_bases[row];
        } else if (bases_by_lane) {
            const int from = r.d >= 0 ? r.d : 0;
            base = __shfl(base_of_rank, from, kWaveSize);
            start = __shfl(start_of_rank, from, kWaveSize);
        } else {
            const int64_t row = int64_t(r.d >= 0 && slot >= 0 ? r.d : 0) * p.tab.chunks_padded;
            base = layout_word(p.tab.rank_bases + row + chunk);
            start = layout_word(p.tab.rank_bases + row);
        }
        if (r.d >= 0 && slot >= 0) {
            r.row_c = base + slot;
            slot = r.row_c - start;             // slot inside the destination bucket
        }
    } else if (r.e >= 0 && slot >= 0) {
        r.row_c = p.slot_is_row ? slot : (r.d > 0 ? p.psum_rank[r.d - 1] : 0) + slot;
    }
    if (first_tile && !p.cached && lane < p.K && p.dst_buffer_slot_idx != nullptr)
        p.dst_buffer_slot_idx[int64_t(t) * p.K + lane] = (r.e >= 0 && slot >= 0) ? p.rank_idx * p.M + slot : -1;
    if (first_tile && !p.cached && p.send_head != nullptr) {
        // V1 handle: wave lane q < R reports the receive row of this token on rank q (-1: not sent there)
        int row_on_rank = -1;
        for (int j = 0; j < p.K; ++j) {
            const int dj = read_lane(r.d, j);
            const int rj = read_lane(r.row_c, j);
            if (dj == lane && rj >= 0) row_on_rank = rj;
        }
        if (lane < p.R) p.send_head[int64_t(t) * p.R + lane] = row_on_rank;
    }

    // Expanded rows of a cached handle are named by the rank's compact row: every valid lane learns it from the master lane.
    if (p.do_expand && p.cached) {
        for (int j = 0; j < p.K; ++j) {
            const int dj = read_lane(r.d, j);
            const int rj = read_lane(r.row_c, j);
            if (r.d >= 0 && dj == r.d && rj >= 0) r.my_row = rj;
        }
    }
    if (p.do_expand && r.e >= 0) {
        if (p.cached) {
            if (r.my_row >= 0 && r.my_row < p.recv_capacity)
                r.erow = p.recv_src_metadata[int64_t(r.my_row) * (p.K + 2) + 2 + lane];
        } else if constexpr (kFused) {
            r.erow = expert_base + epos;
        } else {
            r.erow = layout_word(p.tab.expert_bases + int64_t(chunk) * p.tab.experts_padded + r.e) + epos;
        }
    }
    return r;
}

// Token-level metadata, written once per token (by the wave that owns column tile 0).
//
// What a destination row gets besides its payload goes out in ONE dword store instruction.  Wave lanes take the roles
//   [0, 2K) index dwords | [2K, 3K) weights | [3K, 4K + 2) metadata columns        compact, K <= 15
//   [0, K + 2) metadata columns                                                    expanded
// and a lane's place (a base and a stride by rows) and its word where the row's rank is that of its routing lane, and where not, are
// worked out once: a row then costs an address and a select.  This wavefront's chain is the longest of its token's, and with a branch per
// role and row it was 250 instructions longer at top-8 over 8 ranks.
__device__ __forceinline__ void write_token_metadata(const MoveParams& p, const Route& r, int t, int lane) {
    const int K = p.K;
    uint64_t masters = __ballot(r.row_c >= 0 && r.row_c < p.recv_capacity);
    if (__ballot(r.row_c >= p.recv_capacity) != 0ull && lane == 0) atomicOr(p.status, DEEP_EP_HIP_STATUS_ROW_OVERFLOW);
    if (p.do_expand && p.recv_topk_weights != nullptr && r.erow >= 0 && r.erow < p.expanded_capacity)
        p.recv_topk_weights[r.erow] = r.w;
    if (p.do_expand || 4 * K + 2 <= kWaveSize) {
        int col = p.do_expand ? lane : lane - 3 * K;                              // metadata column (negative: none)
        int src = col - 2;                                                        // routing lane this wave lane reports on
        if (!p.do_expand && lane < 2 * K) src = lane >> 1;
        else if (!p.do_expand && lane < 3 * K) src = lane - 2 * K;
        src = src < 0 || src >= K ? 0 : src;
        const int e_src = __shfl(r.e, src, kWaveSize), d_src = __shfl(r.d, src, kWaveSize);
        const uint32_t w_src = __float_as_uint(__shfl(r.w, src, kWaveSize));
        const int erow_src = p.do_expand ? __shfl(r.erow, src, kWaveSize) : -1;
        uint8_t* base = nullptr;
        uint32_t stride = uint32_t(K) * 4u, match = ~0u, other = ~0u;
        if (!p.do_expand && lane < 2 * K) {
            if (p.recv_topk_idx != nullptr) base = reinterpret_cast<uint8_t*>(p.recv_topk_idx) + lane * 4;
            stride *= 2u;
            match = (lane & 1) ? 0u : uint32_t(e_src - d_src * p.E_l);
        } else if (!p.do_expand && lane < 3 * K) {
            if (p.recv_topk_weights != nullptr) base = reinterpret_cast<uint8_t*>(p.recv_topk_weights) + (lane - 2 * K) * 4;
            match = w_src;
            other = p.zero_nonlocal_w ? 0u : w_src;
        } else if (col < K + 2) {
            stride += 8u;
            if (!p.cached && p.recv_src_metadata != nullptr) base = reinterpret_cast<uint8_t*>(p.recv_src_metadata) + col * 4;
            match = uint32_t(erow_src);
            if (col == 0) {
                match = other = uint32_t(p.rank_idx * p.M + t);
                if (p.recv_src_idx != nullptr) {             // V1: in place of the columns
                    base = reinterpret_cast<uint8_t*>(p.recv_src_idx);
                    stride = 4u;
                    match = other = uint32_t(t);
                }
            }
        }
        // The routing lanes walk the rows with those that store, as they are read from (read_lane): one that has nothing to store itself (V1 without
        // top-k tensors) repeats what the first lane that has stores, the same word to the same place.
        const uint64_t storing = __ballot(base != nullptr);
        if (storing == 0ull) return;
        int rank = d_src;
        if (__ballot(lane < K && base == nullptr) != 0ull) {
            const int like = __builtin_ctzll(storing);
            const uint32_t lo = uint32_t(read_lane(int(uint64_t(base)), like)), hi = uint32_t(read_lane(int(uint64_t(base) >> 32), like));
            const uint32_t its_match = uint32_t(read_lane(int(match), like)), its_other = uint32_t(read_lane(int(other), like));
            const int its_rank = read_lane(d_src, like), its_col = read_lane(col, like), its_stride = read_lane(int(stride), like);
            if (lane < K && base == nullptr) {
                base = reinterpret_cast<uint8_t*>(uint64_t(hi) << 32 | lo);
                stride = uint32_t(its_stride);
                match = its_match;
                other = its_other;
                rank = its_rank;
                col = its_col;
            }
        }
        if (base != nullptr) {
            while (masters) {
                const int j = __builtin_ctzll(masters);
                masters &= masters - 1;
                const uint32_t v = rank == read_lane(r.d, j) ? match : other;
                *reinterpret_cast<uint32_t*>(base + uint64_t(uint32_t(read_lane(r.row_c, j))) * stride) =
                    col == 1 ? uint32_t(p.rank_idx * K + j) : v;
            }
        }
        return;
    }
    while (masters) {
        const int j = __builtin_ctzll(masters);
        masters &= masters - 1;
        const int row = read_lane(r.row_c, j);
        const int dj = read_lane(r.d, j);
        if (lane < K) {
            if (p.recv_topk_idx != nullptr)
                p.recv_topk_idx[int64_t(row) * K + lane] = (r.d == dj) ? int64_t(r.e - dj * p.E_l) : int64_t(-1);
            if (p.recv_topk_weights != nullptr)
                p.recv_topk_weights[int64_t(row) * K + lane] = (p.zero_nonlocal_w && r.d != dj) ? 0.f : r.w;
        }
        if (lane == 0 && p.recv_src_idx != nullptr) p.recv_src_idx[row] = t;
        if (!p.cached && p.recv_src_metadata != nullptr && lane < K + 2) {
            const int v = lane < K ? -1 : lane == K ? p.rank_idx * p.M + t : p.rank_idx * K + j;
            const int col = lane < K ? 2 + lane : lane - K;
            p.recv_src_metadata[int64_t(row) * (K + 2) + col] = v;
        }
    }
}

// Bit mask of lanes that name a destination row, and the row each of them names.
__device__ __forceinline__ uint64_t destination_lanes(const MoveParams& p, const Route& r, int& row_of_lane) {
    if (p.do_expand) {
        row_of_lane = (r.erow >= 0 && r.erow < p.expanded_capacity) ? r.erow : -1;
        if (r.erow >= p.expanded_capacity) atomicOr(p.status, DEEP_EP_HIP_STATUS_ROW_OVERFLOW);
    } else {
        row_of_lane = (r.row_c >= 0 && r.row_c < p.recv_capacity) ? r.row_c : -1;
    }
    return __ballot(row_of_lane >= 0);
}

// Where scale `group` of a (wave-uniform) row goes.  kBlocked: scales_in_blocks.
template <bool kBlocked>
__device__ __forceinline__ uint32_t* scale_place(const MoveParams& p, int row, int group) {
    if constexpr (!kBlocked) return p.recv_sf + (int64_t(row) * p.rsf_ts + int64_t(group) * p.rsf_hs);
    const int r0 = row & ~(kScaleBlockRows - 1);
    const int rows = int(min(p.expanded_capacity - r0, int64_t(kScaleBlockRows)));
    return p.recv_sf + place_in_block((row - r0) * p.num_sf_packs + group, kScaleBlockRows, rows, r0, p.rsf_hs);
}

// ---- single-launch dispatch ----
//
// Grid: C counting workgroups (one 256-token chunk each), one publishing workgroup, then the movers.  A mover cannot
// store a row before the layout is known, and the kernel is bound by its stores, so every microsecond before the
// first store is a microsecond of the launch: the path from the counting workgroups to the movers is kept as short
// as the hardware allows.  A hand-off between workgroups of one launch costs a trip to the memory side for the
// writer's store and one for the reader's load (about a microsecond each on a busy GPU); a flag on top of the data
// would add the writer's wait for its stores, the flag's own trip and a second read.  So the data is its own flag:
//   - every word handed to the movers (chunk totals of the rank buckets, position words, expert bases) carries the
//     tag of this launch in its upper bits (kernels.h) and is stored at agent scope (written through);
//   - a mover workgroup reads what it needs - each thread four chunk totals, each wavefront the position words of
//     its token, and for the expanded layout the base of each lane's (chunk, expert) - first with ordinary loads that
//     go out before the payload loads (first_look), and, where a word does not show the tag yet, again at agent scope
//     (bounded: second_look, await_tagged_words).  It then works the rank bases out for itself (an exclusive prefix
//     sum over the R x C chunk totals, into LDS);
//   - the publisher waits for the chunk_done flags the counting workgroups raise once their stores are acknowledged,
//     clears them, and writes the per-rank and per-expert outputs of the call while the movers are already moving;
//     for the expanded layout the tagged expert bases go out first.
// The tag is generation + 1, and the generation word is advanced by whichever mover learns that every mover has read
// its words: a mover that is done reading advances its gate (mover m uses gate m % kDispatchGates, each gate a cache
// line of its own, because agent-scope atomics on one address serialise at about 11 ns each); the one that brings
// a gate to its number of movers advances gates_finished; the one that brings that to the number of gates in use
// advances the generation.  Gates and gates_finished wrap to 0 on the last increment, so nothing is reset between
// launches.  No workgroup reads the generation after it has moved: counting workgroups and the publisher read it when
// they start, and the movers' reads cannot complete before those have stored their words.  The launch that uses tag
// kTagPeriod clears the tagged tables and starts over at generation 0, so a word can never show the tag of a launch
// other than the running one.  Counting and publishing workgroups have the lowest workgroup ids and wait for nothing
// that is dispatched after them, so every wait ends; each is bounded anyway and reports
// DEEP_EP_HIP_STATUS_LAYOUT_TIMEOUT.
constexpr unsigned kLayoutSpinLimit = 1u << 22;      // polls (each with a short sleep) before giving up: seconds

// The tag of the running launch.  An ordinary (cached) load: the generation word does not change while anyone reads it -
// it is advanced only after every mover has read its tagged words, which it cannot do without the tag - and with tens of
// thousands of wavefronts asking, a read that went to memory every time would make the word's memory channel a hot spot.
__device__ __forceinline__ uint32_t launch_tag(const uint32_t* generation) {
    return (*generation + 1u) << kTagShift;
}

__device__ __forceinline__ uint64_t load_agent64(const void* p) {
    return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ unsigned movers_of_gate(const MoveParams& p, unsigned gate) {
    return (p.num_movers + unsigned(kDispatchGates) - 1u - gate) / unsigned(kDispatchGates);
}

__device__ __forceinline__ void fused_count_block(const MoveParams& p) {
    extern __shared__ uint64_t count_lds[];
    const int c = int(blockIdx.x);
    count_chunk(p.lay, c, p.count_blocks, count_lds);
    wait_for_own_stores();
    __syncthreads();
    if (threadIdx.x == 0) store_agent(p.chunk_done + c, 1);      // for the publisher
}

// All flags[0..n) set?  Polls (bounded), then clears them for the next launch.  Every thread must call it.
__device__ __forceinline__ void await_and_clear_flags(const MoveParams& p, int32_t* flags, int n) {
    bool complete = true;
    for (int i = threadIdx.x; i < n; i += kThreads) {
        unsigned polls = 0;
        while (load_agent(flags + i) == 0 && polls < kLayoutSpinLimit) {
            __builtin_amdgcn_s_sleep(1);
            ++polls;
        }
        if (polls == kLayoutSpinLimit) complete = false;
        store_agent(flags + i, 0);
    }
    if (!complete) atomicOr(p.status, DEEP_EP_HIP_STATUS_LAYOUT_TIMEOUT);
    __syncthreads();
}

__device__ __forceinline__ void finish_hand_off(const MoveParams& p, bool done, uint32_t tag);

// The publisher of an expanded dispatch has read the launch's tag and stored its tagged words (the expert bases): once
// every thread's stores are acknowledged it reports as a party of the hand-off.  Without this a publisher that starts
// late could read the generation after the movers - which wait only for the bases they need, none if no lane is valid -
// have advanced it, and stamp its words with the next launch's tag; and the clearing of the tables at the end of a tag
// period could overtake stores of words no mover waits for.  All threads call it.
__device__ __forceinline__ void publisher_is_done_with_the_tag(const MoveParams& p, uint32_t tag) {
    wait_for_own_stores();
    __syncthreads();
    if (threadIdx.x < kWaveSize) finish_hand_off(p, true, tag);
}

__device__ __forceinline__ void fused_publish_block(const MoveParams& p) {
    extern __shared__ uint64_t count_lds[];
    const PublishLds lds = carve_publish_lds(reinterpret_cast<int*>(count_lds), p.R, p.E);
    const LayoutTables& tab = p.lay.tab;
    const uint32_t tag = launch_tag(p.generation);
    int32_t* tagged_bases = reinterpret_cast<int32_t*>(p.tagged_expert);

    // The movers of an expanded dispatch are waiting for the expert base table, which therefore goes out before
    // anything else, from the tagged chunk totals as they arrive.
    const bool bases_first = p.do_expand && p.E <= kThreads && p.count_blocks <= 32;
    if (bases_first) {
        const bool complete = write_expert_bases_from_registers<kThreads>(tab, p.tagged_expert_counts, tagged_bases, tag, kLayoutSpinLimit,
                                                                          p.R, p.E, p.pub.A, p.count_blocks, lds);
        if (!complete && threadIdx.x == 0) atomicOr(p.status, DEEP_EP_HIP_STATUS_LAYOUT_TIMEOUT);
        publisher_is_done_with_the_tag(p, tag);
    }

    // Everything else waits until the counting workgroups have flagged that their stores are acknowledged.  The expert
    // table (a row per chunk: one writer per cache line, and this workgroup has not touched it before) is then read
    // with ordinary loads, the rank table (lines shared by the writers of 16 chunks) at agent scope.
    await_and_clear_flags(p, p.chunk_done, p.count_blocks);
    sum_expert_columns<kThreads>(tab, p.R, p.E, p.count_blocks, lds.totals);
    publish_experts<kThreads>(p.pub, lds, status_for_host(p.pub));
    if (p.do_expand && !bases_first) {
        __syncthreads();
        write_expert_bases<kThreads, true>(tab, tagged_bases, tag, p.E, p.count_blocks, lds);
        publisher_is_done_with_the_tag(p, tag);
    }
    __syncthreads();
    scan_rank_counts<kThreads>(p.pub, tab, p.R, lds);
}

// What a mover reads of the layout before the layout is known to be there: issued ahead of the payload loads, so
// that a mover that starts after the layout is complete (most of them) has paid no extra trip for it.  Ordinary
// loads, which this XCD's L2 may answer: a word that shows the tag of this launch is this launch's word wherever it
// was cached, and one that does not is read again at agent scope.
struct FirstLook {
    uint64_t totals_lo, totals_hi;     // this thread's four chunk totals
    uint32_t position;                 // this lane's position word
};

__device__ __forceinline__ FirstLook first_look(const MoveParams& p, int t, int lane, bool has_work) {
    FirstLook f{0, 0, 0};
    const int begin = int(threadIdx.x) * 4;
    if (begin < p.R * p.tab.chunks_padded) {
        const vec16 v = load16(p.tagged_rank + begin);
        f.totals_lo = uint64_t(v.x) | (uint64_t(v.y) << 32);
        f.totals_hi = uint64_t(v.z) | (uint64_t(v.w) << 32);
    }
    if (has_work && lane < p.K) f.position = p.pos[int64_t(t) * p.K + lane];
    return f;
}

// The same words read again at agent scope, by a wavefront whose first look came back without the layout: issued before
// the wavefront turns to converting its tile, so that the answer travels while it computes.
__device__ __forceinline__ FirstLook second_look(const MoveParams& p, int t, int lane, bool has_work) {
    FirstLook f{0, 0, 0};
    const int begin = int(threadIdx.x) * 4;
    if (begin < p.R * p.tab.chunks_padded) {
        f.totals_lo = load_agent64(p.tagged_rank + begin);
        f.totals_hi = load_agent64(p.tagged_rank + begin + 2);
    }
    if (has_work && lane < p.K) f.position = uint32_t(load_agent(reinterpret_cast<const int*>(p.pos) + int64_t(t) * p.K + lane));
    return f;
}

// Has this wavefront's first look found everything it asked for?  (Wave-uniform.)
__device__ __forceinline__ bool look_is_complete(const MoveParams& p, const FirstLook& look, uint32_t tag, bool has_work, int lane) {
    bool ok = !(has_work && lane < p.K) || has_tag(look.position, tag);
    if (int(threadIdx.x) * 4 < p.R * p.tab.chunks_padded)
        ok = ok && has_tag(uint32_t(look.totals_lo), tag) && has_tag(uint32_t(look.totals_lo >> 32), tag) &&
             has_tag(uint32_t(look.totals_hi), tag) && has_tag(uint32_t(look.totals_hi >> 32), tag);
    return __all(ok);
}

__device__ __forceinline__ bool totals_tagged(uint64_t lo, uint64_t hi, uint32_t tag) {
    return has_tag(uint32_t(lo), tag) && has_tag(uint32_t(lo >> 32), tag) && has_tag(uint32_t(hi), tag) && has_tag(uint32_t(hi >> 32), tag);
}

// Every mover workgroup works the rank bases out for itself, into its LDS: the exclusive prefix sum over the flattened
// [rank][chunk] table of chunk totals, of which thread i brings entries 4i .. 4i + 3 (tags still on).  `complete`: this
// thread's waits all ended well.  All threads; ends with a barrier.  Returns whether every thread's did.
__device__ __forceinline__ bool build_rank_bases(const MoveParams& p, uint64_t lo, uint64_t hi, bool complete, const int*& bases_out) {
    extern __shared__ uint64_t count_lds[];
    int* bases = reinterpret_cast<int*>(count_lds);
    const int flat = p.R * p.tab.chunks_padded;           // a multiple of 4: a thread's entries share a row
    int* scan_tmp = bases + flat;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int begin = tid * 4;
    const int v0 = int(uint32_t(lo) & kTagValueMask), v1 = int(uint32_t(lo >> 32) & kTagValueMask);
    const int v2 = int(uint32_t(hi) & kTagValueMask), v3 = int(uint32_t(hi >> 32) & kTagValueMask);
    const int sum = v0 + v1 + v2 + v3;
    const int inc = wave_inclusive_sum_by_shuffles(sum);
    if (lane == kWaveSize - 1) scan_tmp[wave] = inc;
    const int all_complete = __syncthreads_and(complete ? 1 : 0);
    int run = inc - sum;
    for (int w = 0; w < wave; ++w) run += scan_tmp[w];
    if (begin < flat) {
        bases[begin] = run;
        bases[begin + 1] = run + v0;
        bases[begin + 2] = run + v0 + v1;
        bases[begin + 3] = run + v0 + v1 + v2;
    }
    __syncthreads();
    bases_out = bases;
    return all_complete != 0;
}

// The mover workgroup is done reading tagged words: its first thread advances the gate.  The value the gate had is
// looked at a little later (settle_gate), after the rows have been resolved and the tile converted, so that most of
// the atomic's round trip is covered.
__device__ __forceinline__ unsigned advance_gate(const MoveParams& p, unsigned mover) {
    const unsigned gate = mover % unsigned(kDispatchGates);
    return atomicInc(p.gates + gate * kDispatchGateStride, movers_of_gate(p, gate) - 1u);
}

// Parties of a launch's hand-off: the gates in use and, for the expanded layout, the publishing workgroup, which reads
// the tag and stores tagged words (the expert bases) itself.
__device__ __forceinline__ unsigned hand_off_parties(const MoveParams& p) {
    const unsigned gates_in_use = p.num_movers < unsigned(kDispatchGates) ? p.num_movers : unsigned(kDispatchGates);
    return gates_in_use + (p.do_expand ? 1u : 0u);
}

// One party of the hand-off is done with this launch's tag (all lanes of one wavefront; `done` is looked at on the first
// lane): a gate whose movers have all read their tagged words, or the publisher of an expanded dispatch once its tagged
// stores are acknowledged.  The party that completes the count advances the generation: by then every tagged word of
// the launch has been read or acknowledged, and nobody will read the generation word for this launch again.  The launch
// that used the last tag clears the tagged tables first, all lanes together (a third of a megabyte: some 15 us once in
// 16383 launches).
__device__ __forceinline__ void finish_hand_off(const MoveParams& p, bool done, uint32_t tag) {
    const int lane = lane_id();
    int last = 0;
    if (lane == 0 && done) {
        const unsigned parties = hand_off_parties(p);
        last = atomicInc(p.gates_finished, parties - 1u) == parties - 1u ? 1 : 0;
    }
    if (__builtin_amdgcn_readfirstlane(last) == 0) return;
    uint32_t next = tag >> kTagShift;                     // generation + 1
    if (next == kTagPeriod) {
        for (int i = lane * 4; i < p.tagged_words; i += kWaveSize * 4) store16_agent(p.tagged + i, vec16{0, 0, 0, 0});
        wait_for_own_stores();
        next = 0;
    }
    if (lane == 0) store_agent(reinterpret_cast<int*>(p.generation), int(next));
}

// First wavefront of a mover workgroup (all its lanes), right before its payload stores - not after them: a wait for the
// atomic's answer behind the stores would be a wait for their acknowledgements too, with the wavefront and its workgroup's
// resources held that long (8192 x 7168 FP8, side by side on one GPU: 86.0 -> 85.7 us).  `seen` counts on its first lane.  The mover
// that was the last of its gate reports the gate.
__device__ __forceinline__ void settle_gate(const MoveParams& p, unsigned mover, unsigned seen, uint32_t tag) {
    const unsigned gate = mover % unsigned(kDispatchGates);
    finish_hand_off(p, seen == movers_of_gate(p, gate) - 1u, tag);
}

// A wavefront's wait (bounded) for the tagged words its threads want.  Returns whether this thread still misses one.
// While the layout is not there, thousands of wavefronts repeat their reads, and every request of theirs stands in
// front of the counting workgroups' stores somewhere: so a waiting wavefront first watches the one kind of word that
// comes last - the expert base of its first routing lane, else its token's position words: one 32-byte request per
// round - and only when that has arrived reads the rest again, whatever is still missing in one trip per round.
__device__ __forceinline__ bool await_tagged_words(uint32_t tag, bool wants_position, const int* position_at, uint32_t& position,
                                                   bool wants_totals, const uint32_t* totals_at, uint64_t& lo, uint64_t& hi,
                                                   bool wants_base, const int* base_at, uint32_t& base_word, unsigned spin_limit) {
    unsigned polls = 0;
    const uint64_t base_lanes = __ballot(wants_base);
    if (base_lanes != 0) {
        const bool watches = wants_base && lane_id() == __builtin_ctzll(base_lanes);
        while (__any(watches && !has_tag(base_word, tag)) && polls < spin_limit) {
            __builtin_amdgcn_s_sleep(4);
            if (watches) base_word = uint32_t(load_agent(base_at));
            ++polls;
        }
    } else {
        while (__any(wants_position && !has_tag(position, tag)) && polls < spin_limit) {
            __builtin_amdgcn_s_sleep(4);
            if (wants_position && !has_tag(position, tag)) position = uint32_t(load_agent(position_at));
            ++polls;
        }
    }
    bool missing;
    for (;;) {
        const bool no_position = wants_position && !has_tag(position, tag);
        const bool no_totals = wants_totals && !totals_tagged(lo, hi, tag);
        const bool no_base = wants_base && !has_tag(base_word, tag);
        missing = no_position || no_totals || no_base;
        if (!__any(missing) || polls >= spin_limit) break;
        if (polls != 0) __builtin_amdgcn_s_sleep(1);
        if (no_position) position = uint32_t(load_agent(position_at));
        if (no_totals) {
            lo = load_agent64(totals_at);
            hi = load_agent64(totals_at + 2);
        }
        if (no_base) base_word = uint32_t(load_agent(base_at));
        ++polls;
    }
    return missing;
}

// Mover workgroups that run beside a counting or the publishing workgroup on one CU read nothing but the layout until
// the layout is there.  A CU's vector memory pipeline takes the requests of all its wavefronts in order, and the payload
// loads of seven mover workgroups keep it busy for microseconds: stores of a counting workgroup that shares the CU
// queue up behind them (measured: positions issued 3.5 us after the launch on a quiet CU, 6 to 8 us beside prefetching
// movers), and every mover of the launch waits for those stores.  Workgroups are handed to the CUs breadth first -
// workgroup i of a launch starts on CU i % num_cus while the first seven or eight per CU are being placed (read back
// from the hardware id registers on MI355X) - so the neighbours of workgroups 0 .. count_blocks are known by index.
// Should a GPU place workgroups differently, the rule holds back other movers: slower, never wrong.
__device__ __forceinline__ bool shares_cu_with_layout_work(const MoveParams& p) {
    return blockIdx.x % unsigned(p.num_cus) <= unsigned(p.count_blocks) && blockIdx.x < unsigned(p.num_cus) * 8u;
}

// Such a workgroup's wait (bounded; await_layout reports a wait that ran out): repeats the first look until it is complete.
__device__ __forceinline__ void hold_for_layout(const MoveParams& p, uint32_t tag, FirstLook& look, int t, int lane, bool has_work) {
    uint32_t no_base = 0;
    const int begin = int(threadIdx.x) * 4;
    await_tagged_words(tag, has_work && lane < p.K, reinterpret_cast<const int*>(p.pos) + int64_t(t) * p.K + lane, look.position,
                       begin < p.R * p.tab.chunks_padded, p.tagged_rank + begin, look.totals_lo, look.totals_hi, false, nullptr, no_base,
                       p.mover_spin_limit);
}

// Everything a mover wavefront needs from the layout of its own launch.
struct FusedLayout {
    const int* flat_bases;    // LDS: exclusive prefix over the chunk totals of the rank buckets
    uint32_t position;        // this lane's position word (tag included)
    int expert_base;          // expanded layout: first row of (this token's chunk, this lane's expert)
    unsigned gate_seen;       // first thread: what advance_gate returned
    uint32_t tag;
    bool complete;            // false: a wait ran out (status already set); the wavefront stores nothing
};

__device__ __forceinline__ FusedLayout await_layout(const MoveParams& p, unsigned mover, const FirstLook& look, uint32_t tag,
                                                    const RouteInputs& in, int t, int lane, bool has_work) {
    FusedLayout f{nullptr, look.position, 0, 0u, tag, true};
    // What this thread waits for: the position word of its lane, four chunk totals, and for the expanded layout the
    // base of its lane's (chunk, expert).  Whatever is missing is read again, all of it in one trip per round.
    const bool wants_position = has_work && lane < p.K;
    const int* position_at = reinterpret_cast<const int*>(p.pos) + int64_t(t) * p.K + lane;
    const int begin = int(threadIdx.x) * 4;
    const bool wants_totals = begin < p.R * p.tab.chunks_padded;
    uint64_t lo = look.totals_lo, hi = look.totals_hi;
    bool wants_base = false;
    const int* base_at = nullptr;
    uint32_t base_word = 0;
    if (p.do_expand) {
        const int64_t e = p.route_mask != nullptr ? (in.mask_byte != 0 ? int64_t(lane) : int64_t(-1)) : in.raw;
        wants_base = wants_position && e >= 0 && e < p.E;
        base_at = reinterpret_cast<const int*>(p.tagged_expert) + int64_t(t / kLayoutChunk) * p.tab.experts_padded + (wants_base ? int(e) : 0);
        if (wants_base) base_word = uint32_t(*base_at);       // an ordinary load first, as in first_look
    }
    const bool missing = await_tagged_words(tag, wants_position, position_at, f.position, wants_totals, p.tagged_rank + begin, lo, hi,
                                            wants_base, base_at, base_word, p.mover_spin_limit);
    f.expert_base = int(base_word & kTagValueMask);
    const bool complete = build_rank_bases(p, lo, hi, !missing, f.flat_bases);      // ends with a workgroup barrier
    if (threadIdx.x == 0) {
        f.gate_seen = advance_gate(p, mover);
        if (!complete) atomicOr(p.status, DEEP_EP_HIP_STATUS_LAYOUT_TIMEOUT);
    }
    f.complete = complete;
    return f;
}

// Workgroups of a single-launch dispatch a CU holds at a time (six wavefronts per SIMD, one per SIMD and workgroup).
constexpr int kResidentWorkgroupsPerCu = 6;

// While the layout is being counted nothing can be stored, and the movers that are resident at launch can only hold so
// much payload in their registers (25 MB at 8192 x 7168): for several microseconds HBM has little to do.  Those movers
// therefore also ask for the tile of the work item two rounds of residents ahead of their own - loads that land in a
// piece of LDS nobody reads, so they cost no registers - which brings that data into the caches while memory is idle
// (a round ahead or three measured less).  Side by side at 8192 x 7168: 86.8 -> 84.9 us in a hot loop, 82.9 -> 81.4 with a
// freshly written input, 89.8 -> 90.3 after a cache flush; 4096 tokens 48.8 -> 46.2 / 49.4 -> 44.4 / 50.7 -> 50.9; 16384
// tokens 164.0 -> 162.6 / 167.7 -> 166.2 / 168.6 -> 169.2.  Movers beside the counting workgroups stay out of it.
// The loads are issued before the wavefront's own payload loads and return in order, so they have landed by the time
// the wavefront uses its payload.  Returns whether the wavefront issued any.
template <int kPairs>
__device__ __forceinline__ bool warm_next_rounds(const MoveParams& p, unsigned work, int lane) {
    if (p.warm_lds_offset == 0 || blockIdx.x >= unsigned(p.num_cus) * unsigned(kResidentWorkgroupsPerCu) ||
        shares_cu_with_layout_work(p))
        return false;
    const unsigned ahead = work + p.warm_ahead;
    if (ahead >= unsigned(p.T) * unsigned(p.tiles)) return false;
    extern __shared__ uint64_t count_lds[];
    const int t = int(ahead / unsigned(p.tiles));
    const int tile = int(ahead - unsigned(t) * unsigned(p.tiles));
    const uint8_t* src = p.x + int64_t(t) * p.row_bytes;
    uint8_t* landing = reinterpret_cast<uint8_t*>(count_lds) + p.warm_lds_offset + (threadIdx.x >> 6) * 1024;
#pragma unroll
    for (int q = 0; q < kPairs; ++q) {
        const int elem = (tile * kPairs + q) * 1024 + lane * 16;
        if (elem < p.H) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + int64_t(elem) * 2),
                                             (__attribute__((address_space(3))) void*)landing, 16, 0, 0);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + int64_t(elem) * 2 + 16),
                                             (__attribute__((address_space(3))) void*)landing, 16, 0, 0);
        }
    }
    return true;
}

// The same for the pass-through kernel, whose tile is kVecs KB of a row (BF16, 4096 x 7168: 80.3 -> 77.2 us in a hot loop,
// 75.6 -> 74.0 with a freshly written input, 83.3 -> 84.0 after a cache flush; 4600 tokens 92.9 -> 86.0 / 85.9 -> 83.5 / 95.3 -> 91.3).
template <int kVecs>
__device__ __forceinline__ bool warm_next_rounds_of_rows(const MoveParams& p, unsigned work, int lane) {
    if (p.warm_lds_offset == 0 || blockIdx.x >= unsigned(p.num_cus) * unsigned(kResidentWorkgroupsPerCu) ||
        shares_cu_with_layout_work(p))
        return false;
    const unsigned ahead = work + p.warm_ahead;
    if (ahead >= unsigned(p.T) * unsigned(p.tiles)) return false;
    extern __shared__ uint64_t count_lds[];
    const int t = int(ahead / unsigned(p.tiles));
    const int tile = int(ahead - unsigned(t) * unsigned(p.tiles));
    const uint8_t* src = p.x + int64_t(t) * p.row_bytes;
    uint8_t* landing = reinterpret_cast<uint8_t*>(count_lds) + p.warm_lds_offset + (threadIdx.x >> 6) * 1024;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
        const int off = (tile * kVecs + i) * 1024 + lane * 16;
        if (off < p.row_bytes)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + off),
                                             (__attribute__((address_space(3))) void*)landing, 16, 0, 0);
    }
    return true;
}

// ---- alignment padding of the expanded layout ----
//
// The padding rows of an expert lie side by side, so its payload, its weights and, in every column (row), its scales are runs of zeros:
// p.slices workgroups share an expert's evenly.  Workgroup `block` of E * slices; needs the finished layout.
__device__ __forceinline__ void zero_padding_rows(const PadParams& p, const unsigned block) {
    const int e = int(block / unsigned(p.slices)), slice = int(block) - e * p.slices;
    const int cnt = p.num_unaligned[e];
    const int64_t first = p.psum_expert[e];                  // start + actual count
    const int n = int(min(int64_t((cnt + p.A - 1) / p.A * p.A - cnt), p.expanded_capacity - first));
    if (n <= 0) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t vecs = int64_t(n) * (p.out_row_bytes / 16);
    const int64_t share = (vecs + int64_t(p.slices) * kThreads - 1) / (int64_t(p.slices) * kThreads) * kThreads;
    const int64_t end = min((slice + 1) * share, vecs);
    uint8_t* rows = p.recv_x + first * p.out_row_bytes;
    const vec16 zero{0, 0, 0, 0};
    for (int64_t i = slice * share + tid; i < end; i += kThreads) store16(rows + i * 16, zero);
    if (p.recv_sf != nullptr && !p.sf_blocked) {
        // a wavefront to a column, or to a row, whichever is contiguous
        const bool columns = p.rsf_ts == 1;
        const int outer = columns ? p.num_sf_packs : n, inner = columns ? n : p.num_sf_packs;
        const int64_t os = columns ? p.rsf_hs : p.rsf_ts, is = columns ? p.rsf_ts : p.rsf_hs;
        uint32_t* scales = p.recv_sf + first * p.rsf_ts;
        for (int o = slice * kWavesPerBlock + (tid >> 6); o < outer; o += p.slices * kWavesPerBlock)
            for (int i = lane; i < inner; i += kWaveSize) scales[o * os + i * is] = 0u;
    }
    if (p.recv_topk_weights != nullptr && slice == 0)
        for (int i = tid; i < n; i += kThreads) p.recv_topk_weights[first + i] = 0.f;
}

// ---- pass-through payload (BF16, or FP8 with caller-provided scale packs) ----
// kScales: rows may come with scale packs (p.recv_sf).
enum : int { kNoScales = 0, kScalesInPlace = 1, kScalesInBlocks = 2 };

// kCached: what goes through the memory-side cache (cached_side).
enum : int { kNeither = 0, kInput = 1, kRows = 2 };

template <int kVecs, bool kFused, int kScales, int kCached>
__device__ __forceinline__ void dispatch_copy(const MoveParams& p) {
    if constexpr (kFused) {
        if (blockIdx.x <= unsigned(p.count_blocks)) {
            if (blockIdx.x < unsigned(p.count_blocks)) fused_count_block(p);
            else fused_publish_block(p);
            return;
        }
    }
    if constexpr (!kFused) {
        if (blockIdx.x >= p.num_movers) {                   // behind the movers of a call that zeroes its padding
            zero_padding_rows(p.pad, blockIdx.x - p.num_movers);
            return;
        }
    }
    const int lane = threadIdx.x & 63;
    const unsigned mover = blockIdx.x - (kFused ? unsigned(p.count_blocks) + 1u : 0u);
    unsigned block = p.xcd_remap ? xcd_contiguous_block(mover, p.num_movers) : mover;
    // the workgroup of the combine that has this one's number runs on the same XCD (kb_of_wavefront)
    if constexpr (kFused && kCached == kRows)
        if (p.shared_tile && !p.xcd_remap) block = xcd_aligned_block(mover, unsigned(p.count_blocks) + 1u, p.num_movers);
    const unsigned work = wave_work_index(block, kWavesPerBlock);
    const bool has_work = work < unsigned(p.T) * unsigned(p.tiles);
    if (!has_work && !kFused) return;
    const int t = has_work ? int(work / unsigned(p.tiles)) : 0;
    const int tile = has_work ? int(work - unsigned(t) * unsigned(p.tiles)) : 0;
    uint32_t tag = 0;
    FirstLook look{0, 0, 0};
    if constexpr (kFused) {
        tag = launch_tag(p.generation);
        look = first_look(p, t, lane, has_work);
        if (shares_cu_with_layout_work(p)) hold_for_layout(p, tag, look, t, lane, has_work);
    }

    bool warmed = false;
    if constexpr (kFused) warmed = warm_next_rounds_of_rows<kVecs>(p, work, lane);

    // Rows are read and written through a descriptor each, which ends with the row: no address and no branch for each vector.
    vec16 v[kVecs];
    const auto src = buffer_of(p.x + int64_t(t) * p.row_bytes, has_work ? p.row_bytes : 0);
    const int at = tile * (kVecs * 1024) + lane * 16;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) v[i] = buffer_load16_as<kCached != kInput>(src, at + i * 1024);

    // The caller's scale packs ride with tile 0: requested with the payload, once, not per destination row.
    const bool packs = kScales != kNoScales && has_work && tile == 0 && p.recv_sf != nullptr;
    uint32_t pack = 0;
    if (packs && lane < p.num_sf_packs) pack = p.sf[int64_t(t) * p.sf_ts + int64_t(lane) * p.sf_hs];

    const RouteInputs route_in = load_route_inputs(p, t, lane);
    const int* flat_bases = nullptr;
    uint32_t word;
    int expert_base = 0;
    unsigned gate_seen = 0;
    if constexpr (kFused) {
        // Payload and routing inputs are in flight; wait for this launch's layout.
        const FusedLayout f = await_layout(p, mover, look, tag, route_in, t, lane, has_work);
        gate_seen = f.gate_seen;
        if (!has_work || !f.complete) {
            if (warmed) wait_for_own_stores();       // no load may still be on its way into this workgroup's LDS
            if (threadIdx.x < kWaveSize) settle_gate(p, mover, gate_seen, tag);
            return;
        }
        word = f.position;
        flat_bases = f.flat_bases;
        expert_base = f.expert_base;
    } else {
        word = load_position_word(p, t, lane);
    }
    const Route r = resolve_route<kFused>(p, route_in, word, flat_bases, expert_base, t, lane, tile == 0);
    if (tile == 0) write_token_metadata(p, r, t, lane);
    if constexpr (kFused)
        if (threadIdx.x < kWaveSize) settle_gate(p, mover, gate_seen, tag);

    int row_of_lane;
    uint64_t dests = destination_lanes(p, r, row_of_lane);
    while (dests) {
        const int j = __builtin_ctzll(dests);
        dests &= dests - 1;
        const int row = read_lane(row_of_lane, j);
        const auto dst = buffer_of(p.recv_x + int64_t(row) * p.row_bytes, p.row_bytes);
#pragma unroll
        for (int i = 0; i < kVecs; ++i)                       // vectors wholly past the row's end are not issued
            if (i == 0 || (tile * kVecs + i) * 1024 < p.row_bytes) buffer_store16_as<kCached != kRows>(dst, at + i * 1024, v[i]);
        if (packs) {
            if (lane < p.num_sf_packs) *scale_place<kScales == kScalesInBlocks>(p, row, lane) = pack;
            for (int g = lane + kWaveSize; g < p.num_sf_packs; g += kWaveSize)        // rows beyond 8192 channels
                *scale_place<kScales == kScalesInBlocks>(p, row, g) = p.sf[int64_t(t) * p.sf_ts + int64_t(g) * p.sf_hs];
        }
        if (!kFused && p.row_by_row) wait_for_own_stores();
    }
}

// Measurement build only (-DDEEP_EP_HIP_WAVE_STAMPS, a library of its own that bench.py --wave-spans loads): every mover
// wavefront of the fused-cast kernels records when it started, when it had issued its last store and when its stores
// were acknowledged, on the 100 MHz wall clock: the span of a launch's wavefronts beside its launch-to-launch time, the
// lifetime of a wavefront, how long before the end the last one starts.
#ifdef DEEP_EP_HIP_WAVE_STAMPS
constexpr int kMaxStampedWaves = 65536;
__device__ long long wave_stamps[3 * kMaxStampedWaves];
#endif

// ---- fused BF16 -> e4m3 cast: lane owns 16 consecutive channels, 8 lanes own one 128-group ----
template <int kPairs, bool kFused, bool kBlocked>
__device__ __forceinline__ void dispatch_cast(const MoveParams& p) {
    if constexpr (kFused) {
        if (blockIdx.x <= unsigned(p.count_blocks)) {
            if (blockIdx.x < unsigned(p.count_blocks)) fused_count_block(p);
            else fused_publish_block(p);
            return;
        }
    }
    if constexpr (!kFused) {
        if (blockIdx.x >= p.num_movers) {                   // behind the movers of a call that zeroes its padding
            zero_padding_rows(p.pad, blockIdx.x - p.num_movers);
            return;
        }
    }
    const int lane = threadIdx.x & 63;
#ifdef DEEP_EP_HIP_WAVE_STAMPS
    const long long stamp_start = wall_clock64();
#endif
    const unsigned mover = blockIdx.x - (kFused ? unsigned(p.count_blocks) + 1u : 0u);
    const unsigned block = p.xcd_remap ? xcd_contiguous_block(mover, p.num_movers) : mover;
    const unsigned work = wave_work_index(block, kWavesPerBlock);
    const bool has_work = work < unsigned(p.T) * unsigned(p.tiles);
    if (!has_work && !kFused) return;
    const int t = has_work ? int(work / unsigned(p.tiles)) : 0;
    const int tile = has_work ? int(work - unsigned(t) * unsigned(p.tiles)) : 0;
    uint32_t tag = 0;
    FirstLook look{0, 0, 0};
    if constexpr (kFused) {
        tag = launch_tag(p.generation);
        look = first_look(p, t, lane, has_work);
        if (shares_cu_with_layout_work(p)) hold_for_layout(p, tag, look, t, lane, has_work);
    }

    bool warmed = false;
    if constexpr (kFused) warmed = warm_next_rounds<kPairs>(p, work, lane);

    vec16 in[kPairs][2];
    const auto src = buffer_of(p.x + int64_t(t) * p.row_bytes, has_work ? p.row_bytes : 0);
    const int at = tile * (kPairs * 1024) + lane * 16;      // channel, and byte of an output row
    if (p.plain_loads) {
#pragma unroll
        for (int q = 0; q < kPairs; ++q) {
            in[q][0] = buffer_load16_as<false>(src, at * 2 + q * 2048);
            in[q][1] = buffer_load16_as<false>(src, at * 2 + q * 2048 + 16);
        }
    } else {
#pragma unroll
        for (int q = 0; q < kPairs; ++q) {
            in[q][0] = buffer_load16_as<true>(src, at * 2 + q * 2048);
            in[q][1] = buffer_load16_as<true>(src, at * 2 + q * 2048 + 16);
        }
    }

    const RouteInputs route_in = load_route_inputs(p, t, lane);

    vec16 out[kPairs];
    float my_scale = 0.f;   // lane L < 8*kPairs ends up holding the scale of group (tile*kPairs*8 + L)
    auto cast_tile = [&]() {
#pragma unroll
        for (int q = 0; q < kPairs; ++q) {
            const float scale_inv = cast_16_channels(in[q][0], in[q][1], out[q]);
            const float gathered = __shfl(scale_inv, (lane & 7) * 8, kWaveSize);
            if ((lane >> 3) == q) my_scale = gathered;
        }
    };

    const int* flat_bases = nullptr;
    uint32_t word;
    int expert_base = 0;
    unsigned gate_seen = 0;
    bool cast_done = false;
    if constexpr (kFused) {
        // Payload and routing inputs are in flight.  A wavefront whose first look found the layout (any wavefront that
        // starts after the first microseconds of the launch) resolves its rows while the payload arrives, as in a
        // launch of its own.  One that has to wait for the layout converts its tile first: when the layout appears,
        // every resident wavefront of the chip is released at once, and the conversions (a few hundred vector
        // instructions each, eight wavefronts to a SIMD) would otherwise queue up between that moment and the first
        // stores of the launch.
        if (!look_is_complete(p, look, tag, has_work, lane)) {
            look = second_look(p, t, lane, has_work);
            cast_tile();
            cast_done = true;
        }
        const FusedLayout f = await_layout(p, mover, look, tag, route_in, t, lane, has_work);
        gate_seen = f.gate_seen;
        if (!has_work || !f.complete) {
            if (warmed) wait_for_own_stores();       // no load may still be on its way into this workgroup's LDS
            if (threadIdx.x < kWaveSize) settle_gate(p, mover, gate_seen, tag);
            return;
        }
        word = f.position;
        flat_bases = f.flat_bases;
        expert_base = f.expert_base;
    } else {
        word = load_position_word(p, t, lane);
    }
    const Route r = resolve_route<kFused>(p, route_in, word, flat_bases, expert_base, t, lane, tile == 0);
    if (tile == 0) write_token_metadata(p, r, t, lane);
    if (!cast_done) cast_tile();
    if constexpr (kFused)
        if (threadIdx.x < kWaveSize) settle_gate(p, mover, gate_seen, tag);
    const int group = tile * kPairs * 8 + lane;
    const bool owns_scale = lane < kPairs * 8 && group * 128 < p.H;

    int row_of_lane;
    uint64_t dests = destination_lanes(p, r, row_of_lane);
    while (dests) {
        const int j = __builtin_ctzll(dests);
        dests &= dests - 1;
        const int row = read_lane(row_of_lane, j);
        const auto dst = buffer_of(p.recv_x + int64_t(row) * p.H, p.H);
#pragma unroll
        for (int q = 0; q < kPairs; ++q)
            if (q == 0 || (tile * kPairs + q) * 1024 < p.H) buffer_store16_as<true>(dst, at + q * 1024, out[q]);
        if (owns_scale) *scale_place<kBlocked>(p, row, group) = __float_as_uint(my_scale);
    }
#ifdef DEEP_EP_HIP_WAVE_STAMPS
    if (lane == 0 && work < unsigned(kMaxStampedWaves)) {
        const long long issued = wall_clock64();
        wait_for_own_stores();
        long long* at = wave_stamps + size_t(work) * 3;
        at[0] = stamp_start;
        at[1] = issued;
        at[2] = wall_clock64();
    }
#endif
}

// ---- the same move as a persistent kernel with a work queue (tuning.persistent_movers) ----
// One workgroup per compute unit stays resident: a few mover wavefronts and a feeder.  Items (token, column tile) are
// handed out in chunks.  A chunk owns sixteen consecutive tickets of the workgroup's ticket counter (LDS) whatever its
// size; a mover draws a ticket, looks the chunk up in a ring of 64-bit words (chunk number, size, first item) and takes
// item `first + offset`, or draws again if the offset lies past the chunk's size.  It requests the loads of its next item
// - payload tile, top-k id, weight, position word, base row of the destination rank - before it converts and stores the
// current one.  The feeder keeps the ring one chunk ahead of the ticket counter: it asks one global counter for chunks
// (one atomic per chunk; the chunks shrink towards the end so that the workgroups run dry together) and posts them; a
// chunk of size zero ends the workgroup.  A feeder that sees the end reports to a wrapping counter at once - its workgroup
// asks for nothing after that - and the last one to report puts the global counter back to zero for the next launch.
//
// Kept as a measured alternative, not a default: on MI355X (8192 x 7168 FP8, move phase on a finished layout) it takes
// 86-95 us from launch to launch against 81 us for one short-lived wavefront per item.  With a static split of the items
// instead of the queue the same loop took 95-104 us: wavefronts get through their items at very different speeds, and
// the slowest ones set the time.  Whether a looping wavefront waits for the acknowledgement of its own stores before it
// uses the loads it issued ahead made no difference when measured (look-ahead loads issued by hand and waited for by
// count, the stores left in flight).
constexpr int kQueueSlot = 16;               // tickets per chunk
constexpr int kQueueStatic = 2;              // chunks a workgroup owns by index (no atomic)
constexpr int kQueueRing = 16;
constexpr int kQueueCounterLine = 128;       // the gate line (kernels.h) that serves as the global item counter

__device__ __forceinline__ unsigned long long queue_word(unsigned chunk, unsigned size, unsigned base) {
    return ((unsigned long long)(((chunk + 1u) << 8) | size) << 32) | base;
}

// Everything a mover needs of one item, requested together.
template <int kPairs>
struct QueuedItem {
    vec16 in[kPairs][2];
    int64_t raw;         // topk_idx entry of routing lane min(lane, K - 1)
    float w;             // its weight
    uint32_t word;       // its position word
    int base;            // base row of (rank min(lane, R - 1), the token's chunk)
};

template <int kPairs>
__device__ __forceinline__ void load_queued_item(const MoveParams& p, unsigned work, int lane, QueuedItem<kPairs>& item) {
    const int t = int(work / unsigned(p.tiles));
    const int tile = int(work - unsigned(t) * unsigned(p.tiles));
    const int64_t at = int64_t(t) * p.K + min(lane, p.K - 1);
    item.raw = p.topk_idx[at];
    item.word = p.pos[at];
    item.w = p.topk_weights != nullptr ? p.topk_weights[at] : 0.f;
    item.base = layout_word(p.tab.rank_bases + int64_t(min(lane, p.R - 1)) * p.tab.chunks_padded + t / kLayoutChunk);
    const uint8_t* src = p.x + int64_t(t) * p.row_bytes;
#pragma unroll
    for (int q = 0; q < kPairs; ++q) {
        // a segment past the end of the row reads the row's last 32 bytes instead (never stored)
        const int elem = min((tile * kPairs + q) * 1024 + lane * 16, p.H - 16);
        item.in[q][0] = load16_stream(src + int64_t(elem) * 2);
        item.in[q][1] = load16_stream(src + int64_t(elem) * 2 + 16);
    }
}

// Routes, converts and stores one item: resolve_route for the one case this kernel is launched for (compact layout, no
// cached handle, top-k routing, at most 64 ranks), with every word it needs already requested.
template <int kPairs>
__device__ __forceinline__ void finish_queued_item(const MoveParams& p, unsigned work, int lane, const QueuedItem<kPairs>& item,
                                                   int start_of_rank) {
    const int t = int(work / unsigned(p.tiles));
    const int tile = int(work - unsigned(t) * unsigned(p.tiles));
    Route r{-1, -1, -1, -1, -1, lane < p.K ? item.w : 0.f};
    int slot = -1;
    if (lane < p.K) {
        if (item.raw >= 0 && item.raw < p.E) r.e = int(item.raw);
        slot = (item.word & kNoPosition) == kNoPosition ? -1 : int(item.word & kNoPosition);
    }
    if (r.e >= 0) r.d = small_div(r.e, p.rcp_E_l);
    else slot = -1;
    {
        const int from = r.d >= 0 ? r.d : 0;
        const int base = __shfl(item.base, from, kWaveSize);
        const int start = __shfl(start_of_rank, from, kWaveSize);
        if (r.d >= 0 && slot >= 0) {
            r.row_c = base + slot;
            slot = r.row_c - start;             // slot inside the destination bucket
        }
    }
    if (tile == 0 && lane < p.K && p.dst_buffer_slot_idx != nullptr)
        p.dst_buffer_slot_idx[int64_t(t) * p.K + lane] = (r.e >= 0 && slot >= 0) ? p.rank_idx * p.M + slot : -1;
    for (int j = 0; j < p.K; ++j) {
        const int dj = read_lane(r.d, j);
        const int rj = read_lane(r.row_c, j);
        if (r.d >= 0 && dj == r.d && rj >= 0) r.my_row = rj;
    }
    if (tile == 0) write_token_metadata(p, r, t, lane);
    vec16 out[kPairs];
    float my_scale = 0.f;
#pragma unroll
    for (int q = 0; q < kPairs; ++q) {
        const float scale_inv = cast_16_channels(item.in[q][0], item.in[q][1], out[q]);
        const float gathered = __shfl(scale_inv, (lane & 7) * 8, kWaveSize);
        if ((lane >> 3) == q) my_scale = gathered;
    }
    const int group = tile * kPairs * 8 + lane;
    const bool owns_scale = lane < kPairs * 8 && group * 128 < p.H;
    int row_of_lane;
    uint64_t dests = destination_lanes(p, r, row_of_lane);
    while (dests) {
        const int j = __builtin_ctzll(dests);
        dests &= dests - 1;
        const int row = read_lane(row_of_lane, j);
        uint8_t* dst = p.recv_x + int64_t(row) * p.H;
#pragma unroll
        for (int q = 0; q < kPairs; ++q) {
            const int elem = (tile * kPairs + q) * 1024 + lane * 16;
            if (elem < p.H) store16_stream(dst + elem, out[q]);
        }
        if (owns_scale) p.recv_sf[int64_t(row) * p.rsf_ts + int64_t(group) * p.rsf_hs] = __float_as_uint(my_scale);
    }
}

template <int kPairs, int kQueueThreads>
__global__ __launch_bounds__(kQueueThreads) void dispatch_cast_queue_kernel(const MoveParams p) {
    constexpr int kQueueWaves = kQueueThreads / kWaveSize;
    __shared__ unsigned ticket;
    __shared__ unsigned long long ring[kQueueRing];
    const int lane = threadIdx.x & 63;
    const unsigned total = unsigned(p.T) * unsigned(p.tiles);
    const unsigned static_items = gridDim.x * unsigned(kQueueStatic * kQueueSlot);
    uint32_t* counter = p.gates + kQueueCounterLine * kDispatchGateStride;
    if (threadIdx.x < kQueueRing) {
        const unsigned c = threadIdx.x;
        unsigned long long word = 0ull;
        if (c < unsigned(kQueueStatic)) {
            const unsigned base = (blockIdx.x * unsigned(kQueueStatic) + c) * unsigned(kQueueSlot);
            word = queue_word(c, base < total ? min(unsigned(kQueueSlot), total - base) : 0u, base);
        }
        ring[c] = word;
        if (c == 0) ticket = 0u;
    }
    __syncthreads();

    if ((threadIdx.x >> 6) == kQueueWaves - 1) {
        // ---- the feeder (one lane) ----
        if (lane != 0) return;
        unsigned posted = kQueueStatic;
        bool ended = (blockIdx.x * unsigned(kQueueStatic) + unsigned(kQueueStatic) - 1u) * unsigned(kQueueSlot) >= total;
        unsigned size = kQueueSlot;
        unsigned polls = 0;
        while (!ended) {
            const unsigned drawing = __hip_atomic_load(&ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) / unsigned(kQueueSlot);
            if (posted > drawing + 1u) {                    // the chunk being drawn and one more are there
                __builtin_amdgcn_s_sleep(8);
                if (++polls > (1u << 26)) {                 // movers that never draw again: give up, and say so
                    atomicOr(p.status, DEEP_EP_HIP_STATUS_LAYOUT_TIMEOUT);
                    break;
                }
                continue;
            }
            const unsigned base = static_items + atomicAdd(counter, size);
            if (base >= total) {
                __hip_atomic_store(&ring[posted % kQueueRing], queue_word(posted, 0u, total), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                ended = true;
            } else {
                __hip_atomic_store(&ring[posted % kQueueRing], queue_word(posted, min(size, total - base), base), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
                ++posted;
                const unsigned left = total - base;
                size = left > total / 4u ? 16u : left > total / 16u ? 8u : 4u;
            }
        }
        if (atomicInc(p.gates_finished, gridDim.x - 1u) == gridDim.x - 1u) atomicExch(counter, 0u);
        return;
    }

    // ---- a mover ----
    // The wavefront's next item, or `total` for none.
    auto draw = [&]() {
        for (;;) {
            unsigned n = 0;
            if (lane == 0) n = __hip_atomic_fetch_add(&ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            n = unsigned(__builtin_amdgcn_readfirstlane(int(n)));
            const unsigned c = n / unsigned(kQueueSlot), o = n % unsigned(kQueueSlot);
            unsigned long long word;
            unsigned spins = 0;
            for (;;) {
                word = __hip_atomic_load(&ring[c % kQueueRing], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (unsigned(word >> 40) == c + 1u) break;
                __builtin_amdgcn_s_sleep(2);
                if (++spins > (1u << 24)) {                 // a feeder that makes no progress, or a slot that went on to a later chunk
                    if (lane == 0) atomicOr(p.status, DEEP_EP_HIP_STATUS_LAYOUT_TIMEOUT);
                    return total;
                }
            }
            const unsigned size = unsigned(word >> 32) & 0xffu;
            if (size == 0u) return total;
            if (o < size) return unsigned(word) + o;
        }
    };

    unsigned work = draw();
    if (work >= total) return;
    const int start_of_rank = layout_word(p.tab.rank_bases + int64_t(min(lane, p.R - 1)) * p.tab.chunks_padded);
    QueuedItem<kPairs> cur;
    load_queued_item<kPairs>(p, work, lane, cur);
    for (;;) {                                              // every mover leaves through the first branch
        const unsigned next = draw();
        if (next >= total) {
            finish_queued_item<kPairs>(p, work, lane, cur, start_of_rank);
            return;
        }
        QueuedItem<kPairs> ahead;
        load_queued_item<kPairs>(p, next, lane, ahead);
        finish_queued_item<kPairs>(p, work, lane, cur, start_of_rank);
        cur = ahead;
        work = next;
    }
}

// The kernels.  The single-launch forms also hold the counting and publishing code, whose register needs must not cost
// the movers their occupancy: they are held to six wavefronts per SIMD (80 registers) - six workgroups per CU, which
// is also where the move streams fastest (more were slower when tried with a leaner counting step, fewer are slower too).
template <int kVecs, int kScales, int kCached>
__global__ __launch_bounds__(kThreads) void dispatch_copy_kernel(const MoveParams p) {
    dispatch_copy<kVecs, false, kScales, kCached>(p);
}
template <int kVecs, int kScales, int kCached>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(6, 8))) void dispatch_copy_single_launch_kernel(const MoveParams p) {
    dispatch_copy<kVecs, true, kScales, kCached>(p);
}
template <int kPairs, bool kBlocked>
__global__ __launch_bounds__(kThreads) void dispatch_cast_kernel(const MoveParams p) {
    dispatch_cast<kPairs, false, kBlocked>(p);
}
template <int kPairs, bool kBlocked>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(6, 8))) void dispatch_cast_single_launch_kernel(const MoveParams p) {
    dispatch_cast<kPairs, true, kBlocked>(p);
}

// Loads the scales of a block (kernels.h) and leaves them in LDS as [row][G + 1].  kBatch loads of a thread are in flight at once, and
// `meanwhile` runs behind the first of them: a workgroup of the pad kernel has one block, and what it costs is its trips to memory.  With one
// load at a time in front of its LDS store the pad kernel took 17.1 us at 2048 x 12288 top-4 of 64 experts and 51 at 4096 x 16384 top-8 of
// 256 (11.2 and 41.4 with scales stored into their columns by the move); it takes 11.9 and 42.
template <int kBatch, typename Meanwhile>
__device__ __forceinline__ void load_block(const PadParams& p, uint32_t* scales, int rows, int64_t r0, Meanwhile&& meanwhile) {
    const int places = rows * p.num_sf_packs;
    const float rcp_G = 1.0f / float(p.num_sf_packs);
    for (int first = threadIdx.x; first - int(threadIdx.x) < places; first += kBatch * kThreads) {
        uint32_t v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
            v[u] = p.recv_sf[place_in_block(min(first + u * kThreads, places - 1), kScaleBlockRows, rows, r0, p.rsf_hs)];
        if (first < kThreads) meanwhile();
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int i = first + u * kThreads;
            if (i < places) scales[i + small_div(i, rcp_G)] = v[u];
        }
    }
}

// ---- put scales that came in blocks into their columns, and zero the padding rows behind a single launch ----
// Workgroups [0, scale_blocks) turn a block each, those behind them zero rows.
__global__ __launch_bounds__(kThreads) void zero_padding_kernel(const PadParams p, const int scale_blocks) {
    extern __shared__ uint32_t scales[];              // [kScaleBlockRows][G + 1]
    if (int(blockIdx.x) < scale_blocks) {
        __shared__ unsigned long long padding;        // rows of the block that are padding
        const int G = p.num_sf_packs, tid = threadIdx.x;
        const int64_t r0 = int64_t(blockIdx.x) * kScaleBlockRows;
        const int last = p.num_unaligned[p.E - 1];
        const int64_t total = int64_t(p.psum_expert[p.E - 1]) - last + (int64_t(last) + p.A - 1) / p.A * p.A;
        if (r0 >= total) return;
        const int rows = int(min(p.expanded_capacity - r0, int64_t(kScaleBlockRows)));
        if (tid == 0) padding = 0ull;
        __syncthreads();
        const auto note_padding = [&] {
            for (int e = tid; e < p.E; e += kThreads) {
                const int cnt = p.num_unaligned[e];
                const int64_t from = max(int64_t(p.psum_expert[e]) - r0, int64_t(0));
                const int64_t to = min(int64_t(p.psum_expert[e]) + ((cnt + p.A - 1) / p.A * p.A - cnt) - r0, int64_t(kScaleBlockRows));
                if (from < to) atomicOr(&padding, (to == 64 ? ~0ull : (1ull << to) - 1ull) & ~((1ull << from) - 1ull));
            }
        };
        if (rows * G <= 4 * kThreads) load_block<4>(p, scales, rows, r0, note_padding);
        else load_block<8>(p, scales, rows, r0, note_padding);
        __syncthreads();
        const unsigned long long none = padding | (total - r0 < kScaleBlockRows ? ~((1ull << (total - r0)) - 1ull) : 0ull);
        for (int i = tid; i < rows * G; i += kThreads) {
            const int g = rows == kScaleBlockRows ? i / kScaleBlockRows : int(unsigned(i) / unsigned(rows));
            const int r = i - g * rows;
            p.recv_sf[r0 + r + g * p.rsf_hs] = (none >> r) & 1ull ? 0u : scales[r * (G + 1) + g];
        }
        return;
    }
    zero_padding_rows(p, blockIdx.x - unsigned(scale_blocks));
}

// ---- stand-alone per-token cast (identity routing) ----
//
// Rows of whole 16-channel pieces on 16-byte boundaries (every hidden a routing call takes): one wavefront per (token,
// kSegments * 1024 channels), lane = 16 consecutive channels as in the fused cast - two 16-byte loads, one 16-byte store -
// and the scales of the tile in one store instruction.  Bound by memory (2 bytes read, 1 written per channel):
// 4096 x 7168 takes 17.2 us, 5.2 TB/s; channel by channel, with 2-byte loads and byte stores, it took 84.3 us.  The
// output is stored with ordinary stores: it is about to be read again, by the dispatch it was made for.
template <int kSegments>
__global__ __launch_bounds__(kThreads) void cast_rows_kernel(const CastParams p, const int tiles) {
    const int lane = threadIdx.x & 63;
    const unsigned work = wave_work_index(blockIdx.x, kWavesPerBlock);
    if (work >= unsigned(p.T) * unsigned(tiles)) return;
    const unsigned t = work / unsigned(tiles);
    const int tile = int(work - t * unsigned(tiles));
    const uint8_t* src = p.x + int64_t(t) * p.H * 2;
    vec16 in[kSegments][2];
#pragma unroll
    for (int q = 0; q < kSegments; ++q) {
        const int elem = (tile * kSegments + q) * 1024 + lane * 16;
        in[q][0] = vec16{0, 0, 0, 0};
        in[q][1] = vec16{0, 0, 0, 0};
        if (elem < p.H) {
            in[q][0] = load16_stream(src + int64_t(elem) * 2);
            in[q][1] = load16_stream(src + int64_t(elem) * 2 + 16);
        }
    }
    uint8_t* dst = p.out + int64_t(t) * p.H;
    float my_scale = 0.f;        // lane L < 8 * kSegments ends up with the scale of group tile * 8 * kSegments + L
#pragma unroll
    for (int q = 0; q < kSegments; ++q) {
        const int elem = (tile * kSegments + q) * 1024 + lane * 16;
        vec16 out;
        const float scale_inv = cast_16_channels(in[q][0], in[q][1], out);
        const float gathered = __shfl(scale_inv, (lane & 7) * 8, kWaveSize);
        if ((lane >> 3) == q) my_scale = gathered;
        if (elem < p.H) store16(dst + elem, out);
    }
    const int groups = (p.H + 127) / 128;
    const int group = tile * kSegments * 8 + lane;
    if (lane < kSegments * 8 && group < groups) p.scales[int64_t(t) * groups + group] = my_scale;
}

// Any other row length or alignment: channel by channel.
__global__ __launch_bounds__(kThreads) void cast_kernel(const CastParams p) {
    const int lane = threadIdx.x & 63;
    const int groups = (p.H + 127) / 128;
    const int tiles = (p.H + 1023) / 1024;
    const int64_t work = int64_t(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
    if (work >= int64_t(p.T) * tiles) return;
    const int t = int(work / tiles);
    const int tile = int(work - int64_t(t) * tiles);
    const int elem = tile * 1024 + lane * 16;
    const uint16_t* src = reinterpret_cast<const uint16_t*>(p.x) + int64_t(t) * p.H;
    float f[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) f[i] = (elem + i < p.H) ? __uint_as_float(uint32_t(src[elem + i]) << 16) : 0.f;
    const float amax = group_amax<true>(f);       // a NaN in the group reaches its scale, as in the torch recipe
    const float scale = 448.0f / amax;
    const float scale_inv = amax / 448.0f;
    uint8_t* dst = p.out + int64_t(t) * p.H;
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
        const uint32_t packed = pack_e4m3x4(f[i] * scale, f[i + 1] * scale, f[i + 2] * scale, f[i + 3] * scale);
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (elem + i + b < p.H) dst[elem + i + b] = uint8_t(packed >> (8 * b));
    }
    const int group = elem / 128;
    if ((lane & 7) == 0 && group < groups && elem < p.H) p.scales[int64_t(t) * groups + group] = scale_inv;
}

// ---- rows of recv_topk_idx beyond the received ones read -1 (csrc/kernels/legacy/intranode.cu:535-545) ----
__global__ __launch_bounds__(kThreads) void fill_tail_kernel(const FillTailParams p) {
    const int64_t first = int64_t(*p.total_rows) * p.K;
    const int64_t end = p.capacity * p.K;
    for (int64_t i = first + int64_t(blockIdx.x) * kThreads + threadIdx.x; i < end; i += int64_t(gridDim.x) * kThreads)
        p.recv_topk_idx[i] = -1;
}

// An attribute of the current device, asked once per device; `fallback` when the runtime does not answer.
static int device_attribute(hipDeviceAttribute_t attribute, std::atomic<int>* cached, int fallback) {
    constexpr int kMaxDevices = 64;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return fallback;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, attribute, dev) != hipSuccess || n <= 0) n = fallback;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

static int lds_bytes_per_cu() {
    static std::atomic<int> cached[64];
    return device_attribute(hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, cached, 160 * 1024);
}

// Destination rows of a token, on average, if the experts were chosen evenly: what decides how many stores follow a load.
// A V1 call without top-k tensors (a cached one, or one routed by is_token_in_rank) has a lane for every rank instead of
// selections, and as many rows as its outputs hold.  (Taken for selections, 32 lanes over 32 ranks stood for 20 rows a token
// where a top-8 handle has 7: a cached 1024 x 7168 BF16 call took 28.3 us, with the tile of a large call, instead of 24.3.)
static double rows_per_token(const MoveParams& p) {
    if (p.rank_lanes) return std::min(double(p.R), double(p.recv_capacity) / p.T);
    if (p.do_expand) return p.K;
    return distinct_ranks(p.R, p.K);
}

// The bytes of those rows.
static double row_bytes_out(const MoveParams& p) {
    const bool cast = p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8;
    return double(p.T) * (cast ? p.H : p.row_bytes) * rows_per_token(p);
}

static bool is_large_input(const MoveParams& p) { return int64_t(p.T) * p.row_bytes >= (int64_t(64) << 20); }

// Which side of a copy goes through the memory-side cache (256 MB).
// - BF16, up to 110 MB of rows and 240 MB with the padding rows zeroed behind them: the rows, which whoever is next then finds there.
//   Dispatch and combine, us, neither / rows, input just written: 277 x 6072 over 8 ranks (18 MB) 24.0 / 22.0, 1024 x 7168 (77 MB) 54.3 / 40.7,
//   4096 x 2048 top-6 (74 MB) 55.7 / 44.1; with a pass over the rows in between that writes as many 30.9 / 31.6, 66.1 / 65.3, 67.7 / 66.4.  With more
//   padding the rows leave the cache again before they are read.  Top-8, aligned to 128, streaming / rows: 646 x 2136 of 384 experts (210 MB)
//   61.4 / 60.0, 400 x 7168 of 112 (206 MB) 62.8 / 61.6, of 128 (235 MB) 67.2 / 66.5, of 144 (264 MB) 72.2 / 72.2, of 160 (294 MB) 78.0 /
//   84.4, 300 x 7168 of 256 (470 MB) 104.4 / 115.5.
// - BF16, more: the input, which the layer in front has just written; so many rows would drive it and each other out.  Dispatch and
//   combine, us, neither / input: 2600 x 7168 over 8 ranks (198 MB) 103.4 / 96.5, 3400 x 7168 (258 MB) 123.7 / 116.5, 8192 x 7168 (622 MB) 261.7 /
//   261.5, V1 4096 x 7168 150.2 / 141.8, expanded 4096 x 4096 top-8 143.3 / 134.8; with the input just written behind 400 MB of other writes 103.7 /
//   99.4, 125.8 / 118.2, 274.8 / 247.4, 151.5 / 141.5, 143.9 / 137.5; with an input that has left the cache by then 103.3 / 110.1, 125.7 /
//   131.3, 265.4 / 275.7, 153.2 / 159.4, 146.1 / 150.6.
// - FP8: neither.  Cast, dispatch and combine, neither / input / rows: 1024 x 7168 (39 MB) 43.2 / 44.3 / 43.4, 2100 x 7168 (80 MB) 71.0 / 71.4 /
//   69.1, 4096 x 7168 (156 MB) 130.1 / 127.4 / 125.4 with three inputs in turn, 126.9 / - / 129.4 with more.
// - BF16, the input larger than that cache or followed by 150 MB and more of zeroed rows: neither.
//   Input called over and over, 20000 x 7168 (287 MB) 597.7 / 603.0; expanded over 256 experts aligned to 128 rows 4883 x 6728 (220 MB of zeros)
//   309.7 / 313.2, 10714 x 6896 (225 MB) 601.2 / 611.5; over 128 (113 MB) it is 567.3 / 565.9 and, input just written, 580.1 / 552.4.
static int cached_side(const MoveParams& p) {
    if (p.payload != DEEP_EP_HIP_PAYLOAD_BF16) return kNeither;
    const double zeroed = p.zeroed_rows * double(p.row_bytes);
    const bool among_padding = p.do_expand && expanded_rows_in_use(p.expanded_capacity, p.recv_capacity, p.T, p.K, p.E, p.R, p.M) * p.row_bytes > kExpandedBytesInCache;
    if (row_bytes_out(p) <= 110e6 && !among_padding) return kRows;
    return double(p.T) * p.row_bytes <= 256e6 && zeroed < 150e6 ? kInput : kNeither;
}

// A launch of so many workgroups of this tile that they fill `rounds` rounds of eight per CU.
static bool fills_rounds(const MoveParams& p, int tile, int rounds) {
    const int bytes = p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8 ? p.H : p.row_bytes;
    const int64_t wavefronts = int64_t(p.T) * ((bytes + tile * 1024 - 1) / (tile * 1024));
    return wavefronts >= int64_t(compute_units()) * rounds * 8 * kWavesPerBlock;
}

// Large moves on a finished layout: tile, and workgroups a CU holds at a time (0: as many as fit).  Scattered stores stream fastest when not too
// many rows are being written at once: a wavefront writes its tile to every row of its token, so what counts is tile x workgroups x rows a token,
// about 20 KB in a fourth of a CU.  Move and combine together, us, best of 1 KB / 2 KB / 4 KB tiles with the workgroups in brackets, and what
// these calls took before, mostly with five or six workgroups of 1 KB or eight of 4 KB:
//   BF16 past the memory-side cache (cached_side):
//     10967 x 5848 of 8 ranks (5.6 rows) 333.1 (4) / 331.9 (2) / 356.6 (8), before 361.5;   8371 x 5048 204.5 (3) / 204.4 (2) / 208.2 (2), 217.8;
//     6221 x 4488 of 64 ranks (9.3) 255.7 / 249.7 / 249.3 (2 each), 263.6;   from 90 MB of input, up to 5.2 rows, 17335 x 3712 (4.4) 250.2 with
//     three of 2 KB, 261.5 with two, 265.1;   15819 x 6096 (2.7) 247 (8) / 243.3 (3) / 249 (2), 245.1;   two rows, 2 KB without a limit / with five, move and with the combine, 16746 x 8072 of 8
//     166.9, 303.5 / 163.6, 299.7;   of 32 173.8, 314.3 / 166.5, 308.2;   20000 x 3976 of 8 99.8, 178.4 / 94.5, 173.2;   of 64 16746 x 8072 185.6, 333.2 / 174.7, 315.2 (four);   rows of 3 and 4 KB 21387 x 1048 (6.5) 174.0 / 171.9 / 165.2 (2 each), 174.1;
//   - nine and more expanded rows over fewer than 32 ranks in two of 1 KB from 450 MB on, rows that are no whole 64 bytes, in % of two of 2 KB, straight /
//     with a pass in between: 500 MB top-10 -4.2 / -1.3, top-9 -2.7 / +0.5, 700 MB top-10 -1.3 / -1.5, top-9 -2.5 / -0.5, 1 GB top-10 -3.6 / -1.0;   of eight rows level
//     / +2.2, of 350 MB of ten +0.7 / -1.3;   rows of whole 64 bytes, which both halves of a KB then share with nobody, +9 to +20 / +10 to +13 (500 MB, 3424 channels
//     top-8 +19.3 / +13.3, top-10 +10.4 / +11.1);
//   - rows of whole KB, whose wavefronts run more alike, up to 430 MB in four or five workgroups of 1 KB: 6608 x 2048 of 8 ranks (5.9) 67.4 (5) / 68.3
//     (4), 72.4;   2805 x 3072 of 32 (8.0) 57.5 (4) / 57.5 (2), 61.2;   and beyond with each row's stores awaited before the next row's are issued, so that
//     a wavefront has one row under way however long that takes; without / with the wait: 20000 x 4096 of 8 (5.3), move alone, 177.4 (2 of 2 KB) / 170.5
//     (6), before 188.5;   whole passes with a layer's other kernels around them, five without / six with the wait: 32000 x 2048 of 32 ranks (7.2) 403.6 /
//     404.4, before 407.3;   8192 x 7168 of 32 348.4 / 345.3, 346.1;   9800 x 7168 of 16 (7.0) 407.5 / 406.6, 410.6;   16384 x 5120 of 64 (7.6) 532.2 / 530.0,
//     534.9;   13211 x 4096 of 16 353.0 / 348.2, 360.1;   16384 x 7168 of 16 (6.5) 607.0 / 609.9, 611.2;   of 32 685.1 / 686.4, 685.5, with five and
//     the wait 710;   on a handle with the wait, five / six, moves alone and with the combine: 16384 x 7168 of 32 (7.2) 340.0, 646.5 /
//     344.1, 671.1;   of 16 (6.5) 316.1, 587.0 / 300.7, 572.7;   9800 x 7168 of 16 185.7, 353.2 / 178.0, 346.6;   13211 x 4096 of 16 149.8, 280.9 / 141.7, 274.8;   16384 x 5120 of 64
//     260.2, 500.2 / 269.1, 505.5;   30000 x 2048 of 32 181.6, 350.9 / 184.5, 348.1;   with the wait, six / as many as fit, moves and with another pass and the combine: of 8 ranks top-6 (4.4)
//     7118 x 7168 111.8, 345.9 / 105.8, 346.0;   15502 x 5120 160.6, 536.8 / 157.0, 527.1;   on a handle 155.7, 535.6 / 147.8, 521.3;   of 64 top-5 (4.8) on one 10075 x 7168 150.9, 509.7 / 152.6, 491.9;
//     rows of 8 and 16 KB, top-6, in three of 2 KB: 24000 x 4096 of 8 ranks (4.4) 361.4 / 369.9 (6), 373.8;   14000 x 8192 418.2 / 430.7 (6), 450.2;
//     where a token goes to fewer than four rows: 14174 x 8192 (3.3) 348 (8 of 1 KB) / 336.8 (4 of 2 KB), 337.5;   16380 x 7168 (3.6) 353.9 (3 of 2 KB),
//     360.9;   17516 x 3584 (3.7) 204.7 (3 of 2 KB) / 197.8 (8 of 1 KB with the wait), 199.5;   without top-k tensors, moves alone, 8192 x 7168 of 4 ranks
//     (2.7) 73.8 (8 of 1 KB) / 75.2 with the wait, 76.1 (4 of 2 KB);   16384 x 4096 top-4 of 8 (3.3) 102.5 / 99.0 with it, 103.3;
//     expanded 25983 x 2560 top-2 156.2 (8 of 2 KB), 173.4;
//   - a few rows among much padding, whose zeroes are most of the call, come here too and are level: 17 shapes of 60 to 1000 tokens x 7168 or 2048 of 256 to 512 experts
//     aligned to 128, layout, move and padding, with a pass over the rows and a combine behind them or not, -0.2 % with four of 2 KB, -1 to +1 without a limit;
//   - rows of whole KB, BF16 and FP8, over 56 to 64 ranks, top-4, with the wait / three (BF16) or four (FP8) of 2 KB, moves and with the combine: 64 ranks BF16 14282 x 7168 203.2, 361.1 /
//     185.4, 347.8;   12496 x 5120 126.1, 228.7 / 122.8, 228.0;   FP8 28564 x 7168 227.1, 543.3 / 200.7, 526.9;   24993 x 5120 145.7, 348.5 / 135.7, 339.8;   move alone of 500 MB, four shapes,
//     40 ranks +1.3 % by 2 KB, 56 -1.9, 60 -2.6, 63 -2.6, 64 -5.0, 65 (whose lanes read the base of their own rank, as on a handle, not of all) +7.3, 96 +6.0;   of 300 MB level, on a handle +5.8;
//   fused cast, expanded, 8192 x 7168 top-8 315.4 (4) / 312.4 (3), 320.6;   16316 x 4608 403.9 (4) / 393.9 (3), 418.5;   compact, 25585 x 3072 of 32
//     ranks 352.5 (4) / 351.8 (4), 364.5;   8192 x 7168 of 8 200.2 (6) / 199.3 (4), 200.4;   12006 x 5120 top-6 (4.4) 204.4 (8) / 202.9 (5), 205.1;   seven
//     rows and more of whole KB, move alone and with the combine, four of 1 KB / four of 2 KB: 16384 x 7168 of 32 204.2, 530.8 / 212.8, 534.9;   of 64 223.1, 555.4 / 230.8,
//     563.6;   8192 x 7168 of 32 110.6, 268.1 / 115.1, 271.9;   of 64 118.0, 280.8 / 125.5, 293.4;   25585 x 3072 of 32 147.3, 352.6 / 144.4, 358.4;   16384 x 4096 of 32 126.5, 307.6 /
//     131.9, 301.2;   fewer rows or other rows 16384 x 7168 of 16 192.9, 474.5 / 192.4, 470.1;   14000 x 6272 top-10 of 16 176.4, 423.2 / 170.2, 411.8;   with
//     blocked scales, whose rows have no single-dword stores, 8192 x 7168 318.1 (5) / 324.0 (3): left alone;
//   FP8 pairs, expanded, of 210 to 270 MB, top-4 / 6 / 8, against what the smaller tiles' rules take: 4 KB -17.5 / -13.7 / -10.2 %, four of 2 KB -14.3 /
//     -11.9 / -8.7, three -7.6 / -9.7 / -7.7;   of 320 MB 4 KB against three or four of 2 KB -3.9 / -2.5 / -0.6;   24963 x 3584 top-9 505.7 (5) / 495.9 (3) / 496.9 (2), 521.1;   compact, 28277 x 4864 (5.9) 485.8 (8) / 473.2 (3) / 474.1 (2),
//     487.5;   35472 x 3968 (4.4) 438.3 (8) / 427.7 (4) / 437.9 (6), 438.3;   rows of whole KB like those of BF16, move alone, without / with the wait: 16384 x 7168 of 32
//     ranks 174.8 (5) / 175.0 (6), 181.6 (8);   32768 x 2048 103.7 (5) / 102.0 (8), 109.0 (8);   8192 x 7168 of 8 66.9 / 64.9 (8);   20000 x 4096 95.0 / 91.3 (8);
//     12000 x 3072 of 16, top-6 45.3 / 44.2 (8);   4096 x 7168 36.0 / 35.4 (8);   12000 x 5120 of 32 101.9 (4) / 105.1 (6), 105.2.
struct MoveShape {
    int tile, per_cu;
    bool in_turn;        // the stores of a row are awaited before the next row's
};

static bool large_move_shape(const MoveParams& p, MoveShape& q) {
    const int bytes = p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8 ? p.H : p.row_bytes, kb = (bytes + 1023) / 1024;
    const double rows = rows_per_token(p), out = row_bytes_out(p);
    if (p.fused || p.cast_pairs != 0 || p.copy_vecs != 0 || kb < 2 || p.sf_blocked) return false;
    if (p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8) {
        if (out < 220e6 || rows < 3.5) return false;
        if (!p.do_expand && rows >= 7.0 && bytes % 1024 == 0) q = {1, 4, false};
        else q = {2, rows < 5.0 ? 5 : p.do_expand ? 3 : 4, false};
        return true;
    }
    const bool whole = bytes % 1024 == 0, many_ranks_few_rows = p.R >= 56 && p.R <= 64 && rows < 4.5 && out >= 350e6 && !p.cached && !p.rank_lanes;
    if (p.payload == DEEP_EP_HIP_PAYLOAD_FP8) {
        if (p.do_expand && kb >= 3 && rows >= 3.2 && out >= 200e6 && out < 300e6) {
            q = {4, 0, false};
            return true;
        }
        if (rows < 3.2 || out < (whole && !p.do_expand ? 100e6 : 280e6)) return false;
        if (whole && !p.do_expand && many_ranks_few_rows) q = {2, 4, false};
        else if (whole && !p.do_expand) q = {1, rows < 6.0 ? 0 : 6, true};
        else q = {2, rows < 5.0 ? 4 : 3, false};
        return true;
    }
    if (cached_side(p) == kRows || (whole && kb == 2)) return false;
    if (rows < 2.4) {
        q = {2, rows < 1.7 || p.do_expand ? 0 : p.R >= 64 ? 4 : 5, false};
        return whole || kb < 3 || kb > 4;
    }
    if (whole) {
        if (p.rank_lanes && rows < 3.9) q = {1, 0, rows >= 3.0};
        else if (many_ranks_few_rows) q = {2, 3, false};
        else if (rows < 3.9 && (rows < 3.5 || kb >= 8 || out < 430e6)) q = {2, rows < 3.5 || kb < 8 ? 4 : 3, false};
        else if (out < 430e6) q = {1, rows < 6.4 ? 5 : 4, false};
        else if ((kb & (kb - 1)) == 0 && kb >= 8 && rows < 5.0) q = {2, 3, false};
        else q = {1, rows < (p.cached ? 5.0 : 4.5) ? 0 : p.cached && rows >= 7.0 ? 5 : 6, true};
        return true;
    }
    if (kb == 3 || kb == 4) {
        q = {4, 2, false};
        return rows >= 3.2;
    }
    if (p.do_expand && rows >= 9.0 && out >= 450e6 && kb >= 5 && p.R < 32 && bytes % 64 != 0) q = {1, 2, false};
    else q = {2, rows < 4.3 || (rows < 5.2 && double(p.T) * p.row_bytes >= 90e6) ? 3 : 2, false};
    return true;
}

// Column tile of a move launch: 1024-channel segments per wavefront for the fused cast, KB of row per wavefront for
// the pass-through payloads.  A tile of one whose last wavefront of a row would be half idle loses to one of two: 65536
// tokens x 768 BF16 over 16 ranks 152 against 175 us, fused cast of 32768 x 1152 over 32 ranks 82 against 104 us.
//
// FP8 rows of calls that leave the chip half empty take the narrowest tile that still gives a CU no more than eight wavefronts (ten with 2 KB
// tiles): what a wavefront does is a chain, and a shorter one is over sooner.  Layout and move of compact calls, top-8 of 8 ranks, with 1 / 2 / 4 KB
// tiles, us: pairs 128 x 4096 10.5 / 10.7 / 11.0, 128 x 8192 10.8 / 10.9 / 11.2, 512 x 4096 12.9 / 12.8 / 13.2, 1237 x 4096 15.2 / 15.6 / 15.8 (2474
// wavefronts of 2 KB), 512 x 14336 18.3 / 17.6 / 17.5 (3584): left alone; fused cast, 1 / 2 segments, 300 x 7168 18.0 / 18.3, 512 x 2048 16.8 / 17.4,
// 512 x 7168 (3584) 19.2 / 18.9.  Not in a single launch, where neighbours of the counting workgroups wait.
// BF16 rows that stay in the memory-side cache take the tile of the combine (kb_of_wavefront), the smallest calls too; beyond its lines tokens of three rows and more of 4, 8
// or 12 KB take 2 KB, move and combine with 1 / 2 / 4 KB: 4096 x 2048 top-6 38.0 / 38.5 / 43.0;  6000 x 2048 top-4 42.0 / 40.9 / 45.3;  2200 x 6144
// top-4 44.1 / 42.2 / 45.7;  3000 x 4096 expanded top-4 47.6 / 46.2 / 50.6; others the widest: 1400 x 7168 47.1 / 47.5 / 44.9, 3500 x 2560 43.7 /
// 45.7 / 43.7, 9000 x 1400 top-4 45.5 / 45.5 / 43.2.
static int move_tile(const MoveParams& p) {
    MoveShape large{};
    if (large_move_shape(p, large)) return large.tile;
    const double rows = rows_per_token(p);
    const auto wavefronts_per_cu_at_most = [&](int tile, int most) {
        const int bytes = p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8 ? p.H : p.row_bytes;
        return !p.fused && !p.do_expand && int64_t(p.T) * ((bytes + tile * 1024 - 1) / (tile * 1024)) <= int64_t(compute_units()) * most;
    };
    if (p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8) {
        // Two segments (2048 channels) measured best at hidden 7168 and 8 ranks: 92.8 us per dispatch against 93.7 (4
        // segments) and 96.9 (7 segments, one wavefront per token).  With many rows per token one segment is ahead on a
        // finished layout, in calls of four rounds and more (16384 x 7168: 32 ranks 199 against 207 us, 16 ranks 185
        // against 189; but 4096 x 4096 over 32 ranks 4 % behind), and in the expanded layout from two rounds on (8192 x
        // 7168 118 against 124 us, 16384 x 4096 top-8 134 against 139); in a single launch, whose workgroups each work out
        // the row bases, only for the expanded layout of a large call.
        if (p.cast_pairs != 0) return p.cast_pairs;
        if (p.H <= 1024 || wavefronts_per_cu_at_most(1, 8)) return 1;
        if (p.fused) return p.do_expand && is_large_input(p) ? 1 : 2;
        if (p.H * 8 <= (p.H + 1023) / 1024 * 7 * 1024) return 2;
        return (p.do_expand ? fills_rounds(p, 1, 2) : rows >= 5.8 && fills_rounds(p, 1, 4)) ? 1 : 2;
    }
    if (p.copy_vecs != 0) return p.copy_vecs;
    const int kb = (p.row_bytes + 1023) / 1024;
    const bool rows_cached = p.payload == DEEP_EP_HIP_PAYLOAD_BF16 && cached_side(p) == kRows;
    if (rows_cached) {
        const int same = p.fused ? kb_of_wavefront(p.T, p.row_bytes, rows, true, p.v1 != 0) : shared_tile(p.T, p.row_bytes, rows, p.like_single != 0, p.v1 != 0);
        if (same != 0) return same;
    }
    if (wavefronts_per_cu_at_most(1, 8)) return 1;
    if (rows_cached && !p.fused && kb % 4 == 0 && rows >= 3.0) return 2;
    if (kb > 2 && wavefronts_per_cu_at_most(2, 10)) return 2;
    const int widest = kb <= 1 ? 1 : kb <= 2 ? 2 : 4;
    // Small, latency-bound calls: up to 4 KB per wavefront, so that fewer wavefronts repeat the routing work (4096 rows
    // of 4 KB: 19.5 us against 21.1 us with 1 KB tiles).  Calls that write 200 MB and more are bound by their stores.
    // Rows of up to 3 KB then take 2 KB (32768 x 1536 top-8: 8 ranks 97 against 104 us, 64 ranks 133 against 146), wider
    // (whole KB in the expanded layout and in V1 calls without top-k tensors, which write little or nothing beside the rows, 1 KB:
    // 32768 x 1024 top-8 over 8 ranks 119 against 127 us, cached V1 77 against 84) ones 1 KB where a token goes to 3.5 rows and more,
    // 2 KB where it goes to fewer and, below five, over 64 ranks.  At 183 MB (16384 x 2048, 4 of 4 ranks) 2 and 4 KB measured the same.
    if (p.fused || row_bytes_out(p) < 200e6) return widest;
    const bool whole = p.row_bytes * 8 > kb * 7 * 1024;           // no wavefront of 1 KB would be half idle
    if (kb <= 3) return kb == 1 || (p.rank_lanes && rows >= 5.0) || ((p.rank_lanes || p.do_expand) && whole) ? 1 : 2;
    return rows >= (p.rank_lanes ? 2.5 : 3.5) && !(p.R >= 64 && rows < 5.0) ? 1 : 2;
}

// Rows of one KB tile with scale packs: their payload and packs, 32 bytes to a row, are partial lines of as many buckets as there
// are ranks, which the caches merge the better the fewer of them are under way.  A wavefront that waits for the stores of a
// row before it starts the next takes, against none that does (65536 x 1024 top-8): 8 ranks 98.7 us for 102.6, 32 ranks 123
// for 141, 64 ranks 134 for 164; 16384 tokens over 8 ranks 30.5 for 30.9.  Wider rows gain by it over 64 ranks and lose over 8
// (32768 x 4096: 231 us for 246, 162 for 157).
static bool stores_row_by_row(const MoveParams& p) {
    MoveShape large{};
    if (large_move_shape(p, large)) return large.in_turn;
    return !p.fused && p.payload != DEEP_EP_HIP_PAYLOAD_CAST_FP8 && p.recv_sf != nullptr && p.row_bytes <= 1024 &&
           rows_per_token(p) >= 3.5 && fills_rounds(p, 1, 2);
}

// How many workgroups of a move kernel launched on a finished layout a CU should hold at a time (0: as many as fit).
// Scattered stores stream fastest when not too many are under way: the more rows a token has, the more ranks they are spread
// over and the wider they are, the fewer.  What large_move_shape leaves, move phase in us, inputs read from memory, with 8 / 6 / 5 / 4 per CU:
//   fused cast, 8192 x 7168, 8 ranks           81.4 / 80.8 / 80.6 / 82.2;   16384 x 7168, 64 ranks 1 KB 272 / 241 / 228
//   fused cast, expanded, 16384 x 4096 top-8   134 / 139 / 141: left alone;           8192 x 7168 top-8 1 KB 122 / 123 / 121,
//                                              and 2 % of the whole pass with inputs that change
//   BF16, 65536 x 512, 64 ranks top-6, 1 KB    140 / 122 / 118 / 123;       65536 x 256 77 / 83 / 88 / 98 (8 ranks): left alone
//   FP8, 16384 x 7168 top-2 of 8 ranks, 2 KB   63.5 / 67.1 / 66 / 68.4: left alone
// Launches that would not fill two rounds of eight per CU, and copies of less than 200 MB (but for rows of 2 KB over 64 ranks:
// 32768 x 768 top-4, 198 MB, 70 us without, 58 with four), are left alone.
static int move_workgroups_per_cu(const MoveParams& p) {
    if (p.fused) return 0;
    if (p.move_workgroups_per_cu != 0)       // two is the least an LDS share within a workgroup's 64 KB can enforce
        return p.move_workgroups_per_cu >= 8 ? 0 : (p.move_workgroups_per_cu < 2 ? 2 : p.move_workgroups_per_cu);
    MoveShape large{};
    if (large_move_shape(p, large)) return large.per_cu;
    const int tile = move_tile(p);
    if (!fills_rounds(p, tile, 2)) return 0;
    const double rows = rows_per_token(p);
    if (p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8) {
        if (p.do_expand) return rows * p.H >= 40 * 1024 ? 5 : 0;
        return tile == 1 && p.R >= 64 ? 5 : 6;
    }
    const int kb = (p.row_bytes + 1023) / 1024;
    const bool spread = rows >= 5.5 || p.R >= 64;
    if (kb == 2 && p.R >= 64 && !p.rank_lanes) return 4;
    if (row_bytes_out(p) < 200e6 || (p.rank_lanes && kb < 8)) return 0;
    if (kb == 1) return spread && p.row_bytes > 512 && !stores_row_by_row(p) ? 5 : 0;
    if (tile == 2 && kb <= 3) return spread ? 4 : rows >= 3.0 ? 5 : 0;
    if (tile == 2) return rows < (p.payload == DEEP_EP_HIP_PAYLOAD_FP8 && p.R < 64 ? 2.5 : 1.7) ? 0 : 4;
    if (spread) return rows >= 5.8 && kb >= 8 ? 5 : 6;
    return kb * rows >= 40.0 ? 6 : 0;
}

}  // namespace

// The limit is set with LDS the kernel never touches: a share that is just too large for one workgroup more, whatever
// granule the LDS is handed out in.
size_t lds_for_residency(int per_cu) {
    return per_cu == 0 ? 0 : (size_t(lds_bytes_per_cu() / (per_cu + 1)) + 256) & ~size_t(255);
}

namespace {

size_t move_lds_bytes(const MoveParams& p) {
    if (!p.fused) return lds_for_residency(move_workgroups_per_cu(p));
    const size_t publish = publish_lds_bytes(p.R, p.E, kThreads);
    const size_t bitmap = count_lds_bytes(p.R, p.E);
    const size_t bases = (size_t(p.R) * p.tab.chunks_padded + kWavesPerBlock) * sizeof(int);
    const size_t bytes = std::max(bases, std::max(bitmap, publish));
    return p.warm_lds_offset != 0 ? size_t(p.warm_lds_offset) + size_t(kWavesPerBlock) * 1024 : bytes;
}

// Grid: the counting workgroups of a single-launch dispatch come first; those that zero padding rows last.
unsigned move_grid(MoveParams& p, int64_t waves) {
    p.num_movers = unsigned((waves + kWavesPerBlock - 1) / kWavesPerBlock);
    return p.num_movers + (p.fused ? unsigned(p.count_blocks) + 1u : p.pad_blocks);
}

// Single launch: the movers that are resident at launch warm the caches for the round after next (warm_next_rounds).
// Call after move_grid.
void plan_cache_warming(MoveParams& p) {
    p.warm_lds_offset = 0;
    if (!p.fused || p.warm_rounds < 0) return;
    const unsigned first_round = unsigned(p.num_cus) * unsigned(kResidentWorkgroupsPerCu);
    // By default two rounds ahead; launches of one and a half to two rounds warm their second round (3072 x 7168 fused
    // cast: 38.2 -> 36.1 us, 3400 tokens 43.8 -> 40.6 us), shorter ones nothing (2048 tokens: 27.9 -> 28.6 us).
    unsigned rounds = p.warm_rounds > 0 ? unsigned(p.warm_rounds) : 2u;
    if (p.warm_rounds == 0 && uint64_t(p.num_movers) <= 2ull * first_round) {
        if (2ull * p.num_movers <= 3ull * first_round) return;
        rounds = 1u;
    }
    if (uint64_t(p.num_movers) <= uint64_t(rounds) * first_round) return;
    p.warm_lds_offset = unsigned((move_lds_bytes(p) + 1023) & ~size_t(1023));
    p.warm_ahead = rounds * first_round * unsigned(kWavesPerBlock);
}

template <int kVecs, int kCached>
hipError_t launch_copy_cached(const MoveParams& p, unsigned blocks, hipStream_t stream) {
    // Rows without scale packs, in tiles of one and two KB: a kernel without the branch on the packs (6490 x 5408 top-8, expanded 101.2 us with the
    // branch, 97.0 without; 16384 x 7168 of 32 ranks 341.1 / 340.3, 10113 x 6392 226.3 / 226.9).  Tiles of four KB have the one with it (8192 x 2048 top-2 21.9 us
    // without the branch, 20.5 with it).
    constexpr int kPlain = kVecs <= 2 ? kNoScales : kScalesInPlace;
    const bool plain = kPlain == kNoScales && p.recv_sf == nullptr;
    auto kernel = p.fused ? (plain ? dispatch_copy_single_launch_kernel<kVecs, kPlain, kCached> : dispatch_copy_single_launch_kernel<kVecs, kScalesInPlace, kCached>)
                          : (plain ? dispatch_copy_kernel<kVecs, kPlain, kCached> : dispatch_copy_kernel<kVecs, kScalesInPlace, kCached>);
    if constexpr (kVecs <= 4 && kCached == kNeither)            // scales come with FP8 rows
        if (p.sf_blocked) kernel = p.fused ? dispatch_copy_single_launch_kernel<kVecs, kScalesInBlocks, kCached> : dispatch_copy_kernel<kVecs, kScalesInBlocks, kCached>;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), move_lds_bytes(p), stream, p);
    return hipGetLastError();
}

template <int kVecs>
hipError_t launch_copy(MoveParams p, hipStream_t stream) {
    p.tiles = (p.row_bytes + kVecs * 1024 - 1) / (kVecs * 1024);
    const unsigned blocks = move_grid(p, int64_t(p.T) * p.tiles);
    plan_cache_warming(p);
    if constexpr (kVecs <= 4) {
        switch (cached_side(p)) {
            case kInput: return launch_copy_cached<kVecs, kInput>(p, blocks, stream);
            case kRows: return launch_copy_cached<kVecs, kRows>(p, blocks, stream);
        }
    }
    return launch_copy_cached<kVecs, kNeither>(p, blocks, stream);
}

template <int kPairs>
hipError_t launch_cast(MoveParams p, hipStream_t stream) {
    p.tiles = (p.H + kPairs * 1024 - 1) / (kPairs * 1024);
    const unsigned blocks = move_grid(p, int64_t(p.T) * p.tiles);
    plan_cache_warming(p);
    if constexpr (kPairs <= 2) {
        if (p.fused) {
            const auto kernel = p.sf_blocked ? dispatch_cast_single_launch_kernel<kPairs, true> : dispatch_cast_single_launch_kernel<kPairs, false>;
            hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), move_lds_bytes(p), stream, p);
            return hipGetLastError();
        }
    }
    if (p.fused) return hipErrorInvalidConfiguration;      // the launch plan keeps wider tiles out of the single launch
    if constexpr (kPairs <= 2) {
        if (p.persistent_movers > 0 && !p.cached && !p.do_expand && p.route_mask == nullptr && p.R <= kWaveSize &&
            p.send_head == nullptr && p.H >= 16 && p.gates != nullptr && p.gates_finished != nullptr) {
            const int64_t items = int64_t(p.T) * p.tiles;
            const int64_t wanted = (items + kQueueSlot * kQueueStatic - 1) / (kQueueSlot * kQueueStatic);
            const unsigned grid = unsigned(std::min<int64_t>(wanted, compute_units()));
            if (p.persistent_movers <= 4) hipLaunchKernelGGL((dispatch_cast_queue_kernel<kPairs, 320>), dim3(grid), dim3(320), 0, stream, p);
            else if (p.persistent_movers <= 8) hipLaunchKernelGGL((dispatch_cast_queue_kernel<kPairs, 576>), dim3(grid), dim3(576), 0, stream, p);
            else hipLaunchKernelGGL((dispatch_cast_queue_kernel<kPairs, 1024>), dim3(grid), dim3(1024), 0, stream, p);
            return hipGetLastError();
        }
    }
    auto kernel = dispatch_cast_kernel<kPairs, false>;
    if constexpr (kPairs <= 2)
        if (p.sf_blocked) kernel = dispatch_cast_kernel<kPairs, true>;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kThreads), move_lds_bytes(p), stream, p);
    return hipGetLastError();
}

}  // namespace

int compute_units() {
    static std::atomic<int> cached[64];
    return device_attribute(hipDeviceAttributeMultiprocessorCount, cached, 256);
}

// Mover workgroups launch_dispatch_move would start for p.
static int64_t move_workgroups(const MoveParams& p) {
    const int tile = move_tile(p);
    const int64_t tiles = p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8 ? (p.H + tile * 1024 - 1) / (tile * 1024)
                                                                    : (p.row_bytes + tile * 1024 - 1) / (tile * 1024);
    return (int64_t(p.T) * tiles + kWavesPerBlock - 1) / kWavesPerBlock;
}

// Where the per-workgroup cost of the single-launch protocol (a look at the layout, one atomic, two workgroup barriers) outweighs
// the launch it saves:
// - rows copied as they are, from 64 MB of input on (one launch / two, us; 1 KB tiles, as wide ones do not help there): BF16 16384 x
//   2048 top-2 of 2 ranks 68.5 / 41.9, 4 of 4 ranks 82.5 / 57.8, top-6 of 16 ranks 108 / 91.6; 8192 x 4096 top-2 of 8 ranks 70.8 / 47.8;
//   FP8 16384 x 4096 4 of 4 ranks 86.0 / 57.6 (6144 x 4096 BF16, 50 MB: 43.8 / 46.9);
// - rows copied as they are, from 300 MB of them on (345 MB of rows of up to 4 KB), BF16 unless said:
//   3072 x 7168: 8 ranks 231 MB 59 / 63, 16 ranks 284 MB 71.8 / 71.4, 32 ranks 316 MB 77.0 / 79.0
//   4096 x 7168: 4 of 4 ranks 160 MB 48 / 51, 8 ranks 308 MB 80.5 / 77.7, 16 ranks 378 MB 97 / 90;   12288 x 2048, 8 ranks 264 MB
//   68 / 73, 16 ranks 324 MB 81.3 / 84.7, 32 ranks 361 MB 94 / 94;   FP8 with scales, 12288 x 4096: 8 ranks 264 MB 69 / 74, 16
//   ranks 324 MB 82.7 / 87.4, 32 ranks 361 MB 98 / 98
// - a fused cast whose movers fill a little more than the first round of residents, all of whom wait for the layout: the rest
//   then runs as a round of its own, while seven per CU of a plain move are under way at once.  Top-8, 1600 movers, one / two:
//   2048 channels 8 ranks 33.8 / 30.7, 32 ranks 39.9 / 37.0; 1024 channels 8 ranks 27.6 / 24.3, 32 ranks 31.8 / 27.3; 7168 channels
//   29.3 / 29.7 and 34.7 / 33.6.  1500 movers (2048 channels) 27.1 / 29.6, 1900 36.4 / 37.5; 4 of 4 ranks (2.7 rows) 23.9 / 23.5
//   and with 7168 channels 23.4 / 23.9: left alone;
// - more than 16384 movers of narrow rows, and of a fused cast.
bool move_prefers_finished_layout(const MoveParams& p, int count_blocks) {
    const int64_t movers = move_workgroups(p), round = int64_t(compute_units()) * kResidentWorkgroupsPerCu;
    if (movers > 16384) return true;
    if (p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8)
        return !p.do_expand && rows_per_token(p) >= 4.0 && movers + count_blocks >= round && movers <= round + compute_units();
    return is_large_input(p) || row_bytes_out(p) >= (p.row_bytes > 4096 ? 300e6 : 345e6);
}

MoveChoice choose_move(const MoveParams& p) {
    return {move_tile(p), move_workgroups_per_cu(p), stores_row_by_row(p) ? 1 : 0, cached_side(p)};
}

hipError_t launch_dispatch_move(MoveParams p, hipStream_t stream) {
    if (p.T == 0) return hipSuccess;
    p.rcp_E_l = 1.0f / float(p.E_l);
    p.num_cus = p.fused ? compute_units() : 0;
    const int tile = move_tile(p);
    p.row_by_row = stores_row_by_row(p) ? 1 : 0;
    p.shared_tile = p.payload == DEEP_EP_HIP_PAYLOAD_BF16 && p.copy_vecs == 0 && kb_of_wavefront(p.T, p.row_bytes, rows_per_token(p), p.fused != 0, p.v1 != 0) != 0 ? 1 : 0;
    if (p.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8) {
        switch (tile) {
            case 1: return launch_cast<1>(p, stream);
            case 2: return launch_cast<2>(p, stream);
            case 7: return launch_cast<7>(p, stream);
            case 8: return launch_cast<8>(p, stream);
            default: return launch_cast<4>(p, stream);
        }
    }
    switch (tile) {
        case 1: return launch_copy<1>(p, stream);
        case 2: return launch_copy<2>(p, stream);
        case 4: return launch_copy<4>(p, stream);
        case 7: return launch_copy<7>(p, stream);
        default: return launch_copy<8>(p, stream);
    }
}

// Scales stored into their columns are a partial line for every row that is moved; in blocks they cost a launch behind the move, which
// otherwise zeroes the padding rows itself.  Layout, move and pad kernel in us, columns / blocks, alignment 128:
//   cast         7564 x 5376 10 of 48 (76 K rows, 3.2 M scales) 131.4 / 122.3; 13983 x 3328 4 of 16 (56 K, 1.5 M) 76.4 / 73.3; 5754 x 5376 8 of 16
//                (46 K, 1.9 M) 80.5 / 79.3; short of rows 4984 x 5760 8 of 64 (40 K, 1.8 M) 77.7 / 79.6; 2425 x 6144 10 of 32 (24 K, 1.2 M) 53.0 /
//                58.3; short of scales 11586 x 1664 4 of 64 (46 K, 0.6 M) 40.8 / 42.4; 300 x 7168 8 of 256 (2.4 K) 41.1 / 46.9
//   FP8 pairs    9468 x 6016 4 of 256 (38 K, 1.8 M) 104.4 / 99.3; 9219 x 6400 8 of 16 (74 K, 3.7 M) 138.6 / 133.0; 9043 x 5504 8 of 32 118.3 / 118.1;
//                narrower rows, whose scales one wavefront has all of, 12085 x 4096 8 of 32 (97 K, 3.1 M) 109.5 / 113.5
// Behind a single launch, where the padding rows take that launch too, padding counts: 3000 x 7168 cast 6 of 64, 16 (1.1 M) 50.1 / 49.4; 700 x 7168
// 8 of 128, 128 (1.2 M) 36.7 / 34.2; short of scales 2568 x 3968 8 of 64, 64 (0.76 M), move and pad 29.9 / 31.2; 4096 x 4096 4 of 64, 64 (0.65 M) 38.0 /
// 38.2; short of rows 2000 x 16384 4 of 32, 64 (10 K) 56.0 / 59.5.
bool scales_in_blocks(const MoveParams& m, int alignment) {
    const bool cast = m.payload == DEEP_EP_HIP_PAYLOAD_CAST_FP8;
    const bool tile_known = cast ? m.cast_pairs >= 0 && m.cast_pairs <= 2 : m.copy_vecs >= 0 && m.copy_vecs <= 4 && m.copy_vecs != 3;
    if (!m.do_expand || alignment <= 1 || m.payload == DEEP_EP_HIP_PAYLOAD_BF16 || m.recv_sf == nullptr || m.rsf_ts != 1 ||
        m.rsf_hs < m.expanded_capacity || m.num_sf_packs < 2 || m.num_sf_packs > kMaxBlockedScales || !tile_known)
        return false;
    const int64_t moved = int64_t(m.T) * m.K, rows = moved + int64_t(m.E) * (alignment - 1);
    if (m.fused) return rows * m.num_sf_packs >= 850000 && rows >= 14000;
    if (cast) return moved * m.num_sf_packs >= 1200000 && moved >= 44000;
    return moved * m.num_sf_packs >= 1700000 && moved >= 36000 && m.num_sf_packs > 40;
}

// 32 KB of an expert's largest padding to a workgroup, and no more than about 4096 of them.
int pad_slices(int experts, int alignment, int out_row_bytes) {
    const int64_t wanted = (int64_t(alignment - 1) * out_row_bytes + 32767) / 32768;
    return int(std::max<int64_t>(std::min<int64_t>(wanted, 4096 / experts), 1));
}

hipError_t launch_zero_padding(const PadParams& p, bool rows, hipStream_t stream) {
    const unsigned row_blocks = rows ? unsigned(p.E) * unsigned(p.slices) : 0u;
    const int scale_blocks = p.sf_blocked ? int((p.expanded_capacity + kScaleBlockRows - 1) / kScaleBlockRows) : 0;
    if (row_blocks + unsigned(scale_blocks) == 0) return hipSuccess;
    const size_t lds = p.sf_blocked ? size_t(kScaleBlockRows) * (p.num_sf_packs + 1) * sizeof(uint32_t) : 0;
    hipLaunchKernelGGL(zero_padding_kernel, dim3(row_blocks + unsigned(scale_blocks)), dim3(kThreads), lds, stream, p, scale_blocks);
    return hipGetLastError();
}

hipError_t launch_fill_tail(const FillTailParams& p, hipStream_t stream) {
    if (p.capacity == 0 || p.K == 0) return hipSuccess;
    const int64_t elems = p.capacity * p.K;
    const unsigned blocks = unsigned(elems / kThreads < 1 ? 1 : (elems / kThreads > 1024 ? 1024 : elems / kThreads));
    hipLaunchKernelGGL(fill_tail_kernel, dim3(blocks), dim3(kThreads), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_cast_kernel(const CastParams& p, hipStream_t stream) {
    if (p.T == 0) return hipSuccess;
    const auto grid = [&](int tiles) { return dim3(unsigned((int64_t(p.T) * tiles + kWavesPerBlock - 1) / kWavesPerBlock)); };
    const bool vectors = p.H % 16 == 0 && reinterpret_cast<uintptr_t>(p.x) % 16 == 0 && reinterpret_cast<uintptr_t>(p.out) % 16 == 0;
    const int segments = (p.H + 1023) / 1024;
    if (vectors && int64_t(p.T) * segments < (int64_t(1) << 31)) {
        const int tiles = (segments + 1) / 2;
        if (segments == 1) hipLaunchKernelGGL(cast_rows_kernel<1>, grid(1), dim3(kThreads), 0, stream, p, 1);
        else hipLaunchKernelGGL(cast_rows_kernel<2>, grid(tiles), dim3(kThreads), 0, stream, p, tiles);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(cast_kernel, grid(segments), dim3(kThreads), 0, stream, p);
    return hipGetLastError();
}

}  // namespace deep_ep_hip

#ifdef DEEP_EP_HIP_WAVE_STAMPS
// Copies the stamps of the first `waves` mover wavefronts of the last fused-cast launch to `out` (3 * waves values).
extern "C" int deep_ep_hip_debug_wave_stamps(long long* out, int waves) {
    if (out == nullptr || waves < 0 || waves > deep_ep_hip::kMaxStampedWaves) return 1;
    return int(hipMemcpyFromSymbol(out, HIP_SYMBOL(deep_ep_hip::wave_stamps), size_t(waves) * 3 * sizeof(long long)));
}
#endif
