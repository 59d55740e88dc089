// Dispatch layout for gfx950: one pass over topk_idx produces per-rank / per-expert counts, the
// token->rank membership, and (for dispatch) the deterministic position of every (token, lane)
// inside its destination bucket.
//
// Replaces csrc/kernels/legacy/layout.cu:10-122 (get_dispatch_layout, where every block rescans
// the whole index array) and the notify warps of deep_ep/include/deep_ep/impls/dispatch.cuh:79-258
// (per-rank / per-expert counts, aligned prefix sums, host mailbox).
//
// Design: a chunk is 256 consecutive tokens, one lane per token.  Each wave sets its lane bit in an LDS bitmap word per rank
// and per expert (ds_or_b64), so that
//   count  = popcount(bitmap)                      and
//   position of token t among chunk tokens routed to the same bucket = popcount(bitmap & lanes below t)
// with no ordering-dependent atomics: placement is a pure function of the input.  A call of one or two chunks is counted
// and published by one workgroup.  In larger ones a workgroup owns a chunk, chunk totals go to tables in the workspace,
// and the last workgroup to finish sums them, writes the base tables the move kernel places rows with, and publishes the
// public prefix sums (publish.h).  A single-launch dispatch runs the same two steps inside the move kernel instead, with a
// counting step that fits the registers of its movers (layout_count.h).
#include <algorithm>

#include "device_utils.h"
#include "kernels.h"
#include "layout_count.h"
#include "publish.h"
#include "../../include/deep_ep_hip.h"

namespace deep_ep_hip {

namespace {

constexpr int kThreads = kLayoutChunk;
constexpr int kWaves = kThreads / kWaveSize;          // of a chunk

// ---- V1 handle bookkeeping (csrc/kernels/legacy/intranode.cu:94-125): one workgroup per destination rank counts the
// tokens of each channel (contiguous token range) that go there, then prefix-sums over channels ----
// Reads nothing the layout pass writes, so with a layout launch its workgroups ride behind the counting ones.  A
// wavefront takes a channel, 512 tokens a trip with all eight byte loads of a lane in flight.  At 4096 tokens and
// 8 ranks it took 8.7 us as a launch of its own behind the layout; the layout launch takes 7.9 us with it.
template <int kBlockWaves>
__device__ __forceinline__ void channel_prefix_block(const IntranodePrefixParams& p, const int d, int* channel_counts /* LDS [C] */) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per_channel = (p.T + p.C - 1) / p.C;
    for (int c = wave; c < p.C; c += kBlockWaves) {
        const int begin = min(per_channel * c, p.T), end = min(begin + per_channel, p.T);
        int count = 0;
        for (int first = begin; first < end; first += 8 * kWaveSize) {
            uint8_t member[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) member[u] = p.mask[int64_t(min(first + u * kWaveSize + lane, end - 1)) * p.R + d];
#pragma unroll
            for (int u = 0; u < 8; ++u) count += __popcll(__ballot(member[u] != 0 && first + u * kWaveSize + lane < end));
        }
        if (lane == 0) channel_counts[c] = count;
    }
    __syncthreads();
    if (wave != 0) return;
    int before = 0;
    for (int c0 = 0; c0 < p.C; c0 += kWaveSize) {
        const int c = c0 + lane;
        const int count = c < p.C ? channel_counts[c] : 0;
        const int end = before + wave_inclusive_sum(count);
        if (c < p.C) {
            if (p.recv_channel_prefix_matrix != nullptr) p.recv_channel_prefix_matrix[d * p.C + c] = end - count;
            if (p.channel_prefix_matrix != nullptr) p.channel_prefix_matrix[d * p.C + c] = end;
        }
        before = read_lane(end, kWaveSize - 1);
    }
    // Only this source rank sends in a one-GPU call: the prefix over source ranks steps once, at rank_idx.
    if (p.rank_prefix_matrix != nullptr)
        for (int i = lane; i < p.R; i += kWaveSize) p.rank_prefix_matrix[i * p.R + d] = i >= p.rank_idx ? before : 0;
}

__global__ __launch_bounds__(kThreads) void intranode_prefix_kernel(const IntranodePrefixParams p) {
    extern __shared__ uint64_t bitmap[];
    channel_prefix_block<kWaves>(p, int(blockIdx.x), reinterpret_cast<int*>(bitmap));
}

// Up to so many selections a token there is a kernel for each number of them, of 30 KB; beyond, one for up to 12, 16, 20 and 32.  Layout and a move of
// 16 channels, us, with a kernel for up to 8 (and two chunks in a workgroup each) / its own: 450 tokens top-3 of 64 10.0 / 8.6, top-5 10.4 / 9.2, top-7 10.7 / 9.7;
// 4096 top-3 of 256 12.0 / 11.4, top-7 12.9 / 12.7; 12000 of 32 ranks top-3 17.6 / 16.9, top-5 19.5 / 19.1.
constexpr int kOwnKernels = 10;

// LDS of a counting workgroup: bitmap words [R + E][waves], spare 32-bit words, and the packed words of the buckets' chunks [R + E][chunks].
constexpr int kSpareWords = kWaveSize;

size_t layout_count_lds_bytes(int R, int E, int chunks) {
    return (size_t(R + E) * chunks * kWaves + kSpareWords / 2) * sizeof(uint64_t) + (size_t(R + E) * chunks + 1) / 2 * 8;
}

// Bound by a chain of trips to memory, not by bytes: index loads, totals out, ticket, totals back, outputs.  Only the
// totals (and the flags) are waited for before the ticket; positions are worked out and stored while it is on its way.  A
// call whose tokens one workgroup holds hands its totals over in LDS instead and publishes them before it works out positions.
// A workgroup's wavefronts have a SIMD each and issue an instruction every four to five cycles, so that between the trips the
// launch takes what its instructions take: the kernels are for a number of selections each, with 32-bit words, one position step
// for all lanes, and tables walked with one add a row.  Back-to-back launches, mailbox included, with kernels for up to
// 8 or 12 selections and 64-bit predicates kept across the pass -> now, us: 128 tokens top-2 of 8 5.0 -> 3.5, 256 top-8 of 256 6.3 -> 4.9, 1237 top-9
// of 72 9.3 -> 7.1, 4096 top-8 7.9 -> 7.4, top-9 9.7 -> 7.4, 16384 top-8 over 32 ranks 9.7 -> 8.6, 10922 top-9 of 18, expanded, 11.7 -> 8.2; counts alone
// (V1), 256 top-9 5.4 -> 4.0, 9830 top-10 of 64 7.8 -> 6.2.
// kExact: KMAX selections a token, otherwise up to KMAX.  kHeldChunks: chunks the only workgroup counts, 0 = a workgroup per
// chunk.  kExpertsPerThread: of the publishing step in one trip, 0 = publish_layout.
template <int KMAX, bool kExact, int kHeldChunks, int kExpertsPerThread>
__global__ __launch_bounds__(kThreads * (kHeldChunks > 1 ? kHeldChunks : 1)) void layout_kernel(const LayoutParams p, const IntranodePrefixParams prefix) {
    constexpr int kChunks = kHeldChunks > 1 ? kHeldChunks : 1;       // of this workgroup
    constexpr int kBlockThreads = kThreads * kChunks, kBlockWaves = kWaves * kChunks;
    extern __shared__ uint64_t bitmap[];   // [(R + E)][kBlockWaves]
    __shared__ int is_last;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int groups = int(gridDim.x) - prefix.R;
    if (int(blockIdx.x) >= groups) {
        channel_prefix_block<kBlockWaves>(prefix, int(blockIdx.x) - groups, reinterpret_cast<int*>(bitmap));
        return;
    }
    const int n = p.R + p.E, K = kExact ? KMAX : p.K;
    const int t = int(blockIdx.x) * kBlockThreads + tid;
    const bool active = t < p.T;
    uint32_t* before_wave = reinterpret_cast<uint32_t*>(bitmap + n * kBlockWaves + kSpareWords / 2);      // [n][kChunks]

    // ---- indices: requested first (they are the longest wait of the pass), the bitmap is cleared while they are in flight ----
    // Lanes past the last token read the last one's, and none of theirs counts.
    int64_t raw[KMAX];
    if (p.route_mask != nullptr) {
#pragma unroll
        for (int k = 0; k < KMAX; ++k) raw[k] = active && k < K && p.route_mask[int64_t(t) * K + k] != 0 ? k : -1;
    } else if (p.T > 0) {
        const int64_t* row = p.topk_idx + int64_t(min(t, p.T - 1)) * K;
        if (KMAX % 2 == 0 && kExact && p.vec_idx) {
#pragma unroll
            for (int i = 0; i < KMAX / 2; ++i) {
                const vec16 q = load16(row + 2 * i);
                raw[2 * i] = int64_t(uint64_t(q.x) | (uint64_t(q.y) << 32));
                raw[2 * i + 1] = int64_t(uint64_t(q.z) | (uint64_t(q.w) << 32));
            }
        } else {
#pragma unroll
            for (int k = 0; k < KMAX; ++k) raw[k] = row[min(k, K - 1)];
        }
    }
    for (int i = tid; i < n * kBlockWaves; i += kBlockThreads) bitmap[i] = 0ull;
    __syncthreads();

    // ---- bitmaps ----
    // No predicate outlives its use; a selection that counts nowhere ORs no bit into a spare word of its lane (atomics of one wavefront on one
    // address take turns); for ranks one OR per selection and one ballot per rank.
    uint32_t* words32 = reinterpret_cast<uint32_t*>(bitmap);
    const uint32_t my_bit = 1u << (lane & 31), my_word = uint32_t(tid >> 5), spare = uint32_t(n) * (kBlockWaves * 2) + uint32_t(lane);
    const uint32_t experts = uint32_t(p.E);
    const uint64_t limit = active ? experts : 0u;
    const float rcp_experts_per_rank = 1.0f / float(p.E_l);
    uint32_t e[KMAX];                            // p.E: none
    uint32_t seen = 0;
    int out_of_range = -1;                       // negative: none
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
        const uint32_t lo = uint32_t(raw[k]), hi = uint32_t(uint64_t(raw[k]) >> 32);
        const bool counts = uint64_t(raw[k]) < limit && k < K;
        e[k] = counts ? lo : experts;
        out_of_range &= counts || k >= K ? -1 : int(hi);
        const uint32_t bit = counts ? my_bit : 0u;
        const uint32_t word = counts ? (uint32_t(p.R) + lo) * (kBlockWaves * 2) + my_word : spare;
        seen |= atomicOr(words32 + word, bit) & bit;         // a bit that is set already: the token names the expert twice
    }
    if (p.R <= kBallotRanks) {
        uint32_t ranks = 0;                      // bit r: this token goes to rank r; bit R: nowhere
#pragma unroll
        for (int k = 0; k < KMAX; ++k) ranks |= 1u << small_div(int(e[k]), rcp_experts_per_rank);
        uint64_t mine = 0;
        for (int r = 0; r < p.R; ++r) {
            const uint64_t members = __ballot((ranks >> r) & 1u);
            if (lane == r) mine = members;
        }
        if (lane < p.R) bitmap[lane * kBlockWaves + wave] = mine;
    } else {
#pragma unroll
        for (int k = 0; k < KMAX; ++k) {
            const uint32_t d = uint32_t(small_div(int(e[k]), rcp_experts_per_rank));
            atomicOr(words32 + (e[k] < experts ? d * (kBlockWaves * 2) + my_word : spare), e[k] < experts ? my_bit : 0u);
        }
    }
    int flags = active && out_of_range >= 0 ? DEEP_EP_HIP_STATUS_EXPERT_OUT_OF_RANGE : 0;
    if (p.pos != nullptr && seen != 0) flags |= DEEP_EP_HIP_STATUS_DUPLICATE_EXPERT;
    if (flags != 0) atomicOr(p.status, flags);
    __syncthreads();

    // ---- totals: per bucket and chunk the bits set go out, and those of the wavefronts before each wavefront of the chunk are packed
    // into one LDS word (three 10-bit fields), so that a position costs two independent LDS reads ----
    int* totals = nullptr;                                   // [n][kChunks]
    if constexpr (kHeldChunks > 0)
        totals = reinterpret_cast<int*>(reinterpret_cast<uint8_t*>(bitmap) + p.lds_totals);
    for (int j = tid; j < n * kChunks; j += kBlockThreads) {
        const uint64_t* words = bitmap + j * kWaves;
        const int c0 = __popcll(words[0]), c1 = __popcll(words[1]), c2 = __popcll(words[2]), c3 = __popcll(words[3]);
        before_wave[j] = uint32_t(c0) | (uint32_t(c0 + c1) << 10) | (uint32_t(c0 + c1 + c2) << 20);
        if constexpr (kHeldChunks > 0) {
            totals[j] = c0 + c1 + c2 + c3;
        } else {
            store_agent(j < p.R ? p.tab.rank_counts + int64_t(j) * p.tab.chunks_padded + blockIdx.x
                                : p.tab.expert_counts + int64_t(blockIdx.x) * p.tab.experts_padded + (j - p.R), c0 + c1 + c2 + c3);
        }
    }
    unsigned ticket = 0;
    if constexpr (kHeldChunks > 0) {
        wait_for_own_stores();                               // flags ORed into the status word, if any
        __syncthreads();
        publish_layout_in_one_trip<kBlockThreads, kHeldChunks, kExpertsPerThread>(p.pub, p.tab, kHeldChunks, p.expert_bases != 0, totals, totals + n * kChunks);
    } else {
        const int pad = p.tab.chunks_padded - groups;        // the padding columns of the rank table are cleared by the first workgroup
        if (blockIdx.x == 0)
            for (int i = tid; i < p.R * pad; i += kBlockThreads) store_agent(p.tab.rank_counts + (i / pad) * p.tab.chunks_padded + groups + i % pad, 0);
        // Hand the chunk totals to whichever workgroup finishes last: they were stored at agent scope (written through),
        // so waiting for our own stores is all the release there is - no write-back of the whole L2 - then take a ticket.
        wait_for_own_stores();
        __syncthreads();
        if (tid == 0) ticket = atomicAdd(p.done_counter, 1u);
    }

    // ---- positions and copies: nobody of this launch waits for them ----
    if (active && p.pos != nullptr) {
        // One word per (token, lane): the slot of the token inside its chunk for the lane's destination rank (master lanes
        // only: the last lane that names the rank) and the position of the lane inside its chunk for its expert (kernels.h).
        // Position inside the chunk = bits of this wavefront's word below the lane + bits of the chunk's wavefronts before it.
        const uint64_t below = lanes_below(lane);
        const int wave_of_chunk = wave & (kWaves - 1), chunk_here = wave / kWaves;
        const uint32_t wave_shift = wave_of_chunk > 0 ? 10u * uint32_t(wave_of_chunk - 1) : 0u;
        const uint32_t earlier_bits = wave_of_chunk > 0 ? 10u : 0u;
        auto position = [&](uint32_t bucket) {
            const uint64_t word = bitmap[bucket * kBlockWaves + wave] & below;
            return uint32_t(__popcll(word)) + __builtin_amdgcn_ubfe(before_wave[bucket * kChunks + chunk_here], wave_shift, earlier_bits);
        };
        constexpr uint32_t kNoExpertPosition = kNoPosition << kExpertPositionShift;
        uint32_t packed[KMAX];
        // the lanes are walked backwards with the set of ranks seen so far
        if (p.R < 32) {
            uint32_t later_ranks = 1u << p.R;                // where a selection without an expert would go
#pragma unroll
            for (int k = KMAX - 1; k >= 0; --k) {
                const uint32_t d = uint32_t(small_div(int(e[k]), rcp_experts_per_rank));
                const bool master = __builtin_amdgcn_ubfe(later_ranks, d, 1u) == 0u;
                later_ranks |= 1u << d;
                packed[k] = kNoExpertPosition | (master ? position(d) : kNoPosition);
            }
        } else {
            uint64_t later_ranks = 0;
#pragma unroll
            for (int k = KMAX - 1; k >= 0; --k) {
                const int d = small_div(int(e[k]), rcp_experts_per_rank);
                bool master = e[k] < experts;
                if (p.R <= 64) {
                    const uint64_t rank_bit = master ? 1ull << d : 0ull;
                    master = (rank_bit & ~later_ranks) != 0;
                    later_ranks |= rank_bit;
                } else {
#pragma unroll
                    for (int j = k + 1; j < KMAX; ++j)
                        if (small_div(int(e[j]), rcp_experts_per_rank) == d) master = false;
                }
                const uint32_t at = position(uint32_t(e[k] < experts ? d : 0));
                packed[k] = kNoExpertPosition | (master ? at : kNoPosition);
            }
        }
        if (p.expert_bases) {                                // only the expanded layout places rows by expert
#pragma unroll
            for (int k = 0; k < KMAX; ++k) {
                const uint32_t at = position(e[k] < experts ? uint32_t(p.R) + e[k] : 0u);
                if (e[k] < experts) packed[k] = (packed[k] & kNoPosition) | at << kExpertPositionShift;
            }
        }
        uint32_t* dst = p.pos + int64_t(t) * K;
        if constexpr (KMAX % 4 == 0 && kExact) {
#pragma unroll
            for (int k = 0; k < KMAX; k += 4) store16(dst + k, vec16{packed[k], packed[k + 1], packed[k + 2], packed[k + 3]});
        } else {
#pragma unroll
            for (int k = 0; k < KMAX; ++k)
                if (k < K) dst[k] = packed[k];
        }
    }
    if (active && p.copied_topk_idx != nullptr) {
        int64_t* dst = p.copied_topk_idx + int64_t(t) * K;
#pragma unroll
        for (int k = 0; k < KMAX; ++k)
            if (k < K) dst[k] = raw[k];
    }
    if (active && p.is_token_in_rank != nullptr) {
        for (int r = 0; r < p.R; ++r)
            p.is_token_in_rank[int64_t(t) * p.R + r] = uint8_t((bitmap[r * kBlockWaves + wave] >> lane) & 1ull);
    }

    if constexpr (kHeldChunks == 0) {
        if (tid == 0) is_last = (ticket == unsigned(groups) - 1u) ? 1 : 0;
        __syncthreads();
        if (!is_last) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");

        // ---- last workgroup: per-bucket totals, the public prefix sums and the row bases (LDS is re-carved) ----
        int* lds = reinterpret_cast<int*>(bitmap);
        if constexpr (kExpertsPerThread == 0) publish_layout<kThreads>(p.pub, p.tab, groups, p.expert_bases != 0, lds);
        else publish_layout_in_one_trip<kThreads, 0, kExpertsPerThread>(p.pub, p.tab, groups, p.expert_bases != 0, nullptr, lds);
        if (tid == 0) *p.done_counter = 0u;                // ready for the next launch
    }
}

template <int KMAX, bool kExact>
void launch_layout(const LayoutParams& q, const IntranodePrefixParams& prefix, dim3 grid, size_t lds, int held_chunks, hipStream_t stream) {
    const bool by_one = fits_one_trip(1, q.R, q.E, q.tab.chunks_padded, kThreads), by_two = fits_one_trip(2, q.R, q.E, q.tab.chunks_padded, kThreads);
    auto kernel = held_chunks == 1 ? (by_one ? layout_kernel<KMAX, kExact, 1, 1> : layout_kernel<KMAX, kExact, 1, 2>)
                  : by_one         ? layout_kernel<KMAX, kExact, 0, 1>
                  : by_two         ? layout_kernel<KMAX, kExact, 0, 2>
                                   : layout_kernel<KMAX, kExact, 0, 0>;
    if constexpr (kExact)
        if (held_chunks == 2) kernel = layout_kernel<KMAX, kExact, 2, 1>;
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads * std::max(held_chunks, 1)), lds, stream, q, prefix);
}

}  // namespace

hipError_t launch_intranode_prefix(const IntranodePrefixParams& p, hipStream_t stream) {
    if (p.R == 0 || p.C == 0) return hipSuccess;
    hipLaunchKernelGGL(intranode_prefix_kernel, dim3(p.R), dim3(kThreads), size_t(p.C) * sizeof(int), stream, p);
    return hipGetLastError();
}

hipError_t launch_layout_kernel(const LayoutParams& p, const IntranodePrefixParams& wanted, hipStream_t stream) {
    IntranodePrefixParams prefix = wanted;
    if (prefix.C == 0) prefix.R = 0;
    const int num_chunks = p.T > 0 ? (p.T + kThreads - 1) / kThreads : 1;
    // The counting step's LDS first; the last of several workgroups re-carves it for the publishing step, the only one has its
    // totals and the publishing step's scratch behind it.
    // Two chunks in one workgroup / in one each, us, 450 tokens: top-8 of 256 over 8 ranks 6.4 / 6.8, top-3 of 64 5.2 / 6.7; of more buckets than threads,
    // or with a kernel for up to so many selections, the one workgroup is behind: top-12 of 256 over 64 ranks 12.6 / 10.5, top-16 of 512 17.0 / 13.7.
    const int held_chunks = num_chunks == 1 && p.R <= kThreads && p.E <= 2 * kThreads                      ? 1
                            : num_chunks == 2 && p.K <= kOwnKernels && p.R + p.E <= 320 && p.R <= kThreads ? 2
                                                                                                           : 0;
    const int chunks = std::max(held_chunks, 1);
    LayoutParams q = p;
    q.vec_idx = (reinterpret_cast<uintptr_t>(p.topk_idx) % 16 == 0) ? 1 : 0;
    q.lds_totals = int(layout_count_lds_bytes(p.R, p.E, chunks));
    size_t lds = size_t(q.lds_totals);
    if (held_chunks > 0) lds += (size_t(p.R + p.E) * chunks + publish_scratch_ints(p.R, kThreads * chunks)) * sizeof(int);
    if (held_chunks == 0) lds = std::max(lds, publish_lds_bytes(p.R, p.E, kThreads));
    if (prefix.R != 0) lds = std::max(lds, size_t(prefix.C) * sizeof(int));
    const dim3 grid((held_chunks > 0 ? 1 : num_chunks) + prefix.R);
    const auto launch = [&](auto kernels) { kernels(q, prefix, grid, lds, held_chunks, stream); };
    static_assert(kOwnKernels == 10, "one case for each");
    switch (p.K) {
        case 1: launch(launch_layout<1, true>); break;
        case 2: launch(launch_layout<2, true>); break;
        case 3: launch(launch_layout<3, true>); break;
        case 4: launch(launch_layout<4, true>); break;
        case 5: launch(launch_layout<5, true>); break;
        case 6: launch(launch_layout<6, true>); break;
        case 7: launch(launch_layout<7, true>); break;
        case 8: launch(launch_layout<8, true>); break;
        case 9: launch(launch_layout<9, true>); break;
        case 10: launch(launch_layout<10, true>); break;
        default:
            if (p.K <= 12) launch(launch_layout<12, false>);
            else if (p.K <= 16) launch(launch_layout<16, false>);
            else if (p.K <= 20) launch(launch_layout<20, false>);
            else launch(launch_layout<32, false>);
    }
    return hipGetLastError();
}

}  // namespace deep_ep_hip
