// Dispatch layout for gfx950: one pass over topk_idx produces per-rank / per-expert counts, the
// token->rank membership, and (for dispatch) the deterministic position of every (token, lane)
// inside its destination bucket.
//
// Replaces csrc/kernels/legacy/layout.cu:10-122 (get_dispatch_layout, where every block rescans
// the whole index array) and the notify warps of deep_ep/include/deep_ep/impls/dispatch.cuh:79-258
// (per-rank / per-expert counts, aligned prefix sums, host mailbox).
//
// Design: a workgroup owns a chunk of 256 consecutive tokens (one lane per token).  Each wave sets
// its lane bit in an LDS bitmap word per rank and per expert (ds_or_b64), so that
//   count  = popcount(bitmap)                      and
//   position of token t among chunk tokens routed to the same bucket = popcount(bitmap & lanes below t)
// with no ordering-dependent atomics: placement is a pure function of the input (layout_count.h).  Chunk
// totals go to tables in the workspace; the last workgroup to finish sums them, writes the base tables the
// move kernel places rows with, and publishes the public prefix sums (publish.h).  A single-launch dispatch
// runs the same two steps inside the move kernel instead (dispatch.hip).
#include "device_utils.h"
#include "kernels.h"
#include "layout_count.h"
#include "publish.h"
#include "../../include/deep_ep_hip.h"

namespace deep_ep_hip {

namespace {

constexpr int kThreads = kLayoutChunk;
constexpr int kWaves = kThreads / kWaveSize;

// ---- V1 handle bookkeeping (csrc/kernels/legacy/intranode.cu:94-125): one workgroup per destination rank counts the
// tokens of each channel (contiguous token range) that go there, then prefix-sums over channels ----
// Reads nothing the layout pass writes, so with a layout launch its workgroups ride behind the counting ones.  A
// wavefront takes a channel, 512 tokens a trip with all eight byte loads of a lane in flight.  At 4096 tokens and
// 8 ranks it took 8.7 us as a launch of its own behind the layout; the layout launch takes 7.9 us with it.
__device__ __forceinline__ void channel_prefix_block(const IntranodePrefixParams& p, const int d, int* channel_counts /* LDS [C] */) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per_channel = (p.T + p.C - 1) / p.C;
    for (int c = wave; c < p.C; c += kWaves) {
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
    channel_prefix_block(p, int(blockIdx.x), reinterpret_cast<int*>(bitmap));
}

// Bound by a chain of trips to memory, not by bytes: index loads, totals out, ticket, totals back, outputs.  Only the
// totals (and the flags) are waited for before the ticket; positions and copies are stored while it is on its way.  A
// call of one chunk hands its totals over in LDS instead.  Launch time, mailbox included, with everything
// waited for before the ticket and everything read back -> now: 128 tokens top-2 9.6 -> 6.1 us, 1237 top-9 13.0 -> 9.8,
// 4096 top-8 10.0 -> 8.3, 16384 top-8 over 32 ranks 14.8 -> 11.5.
// kExpertsPerThread: of the publishing step in one trip, 0 = publish_layout.
template <int KMAX, bool kOneChunk, int kExpertsPerThread>
__global__ __launch_bounds__(kThreads) void layout_kernel(const LayoutParams p, const IntranodePrefixParams prefix) {
    extern __shared__ uint64_t bitmap[];   // [(R + E)][kWaves]
    __shared__ int is_last;
    const int tid = threadIdx.x;
    const int num_chunks = int(gridDim.x) - prefix.R;
    if (int(blockIdx.x) >= num_chunks) {
        channel_prefix_block(prefix, int(blockIdx.x) - num_chunks, reinterpret_cast<int*>(bitmap));
        return;
    }
    if constexpr (kOneChunk) {
        int* totals = reinterpret_cast<int*>(bitmap) + count_lds_bytes(p.R, p.E) / sizeof(int);
        count_chunk<KMAX, false>(p, 0, 1, bitmap, totals, [&] {
            wait_for_own_stores();                         // flags ORed into the status word, if any
            __syncthreads();
            publish_layout_in_one_trip<kThreads, true, kExpertsPerThread>(p.pub, p.tab, 1, p.expert_bases != 0, totals, totals + p.R + p.E);
        });
    } else {
        // Hand the chunk totals to whichever workgroup finishes last: they were stored at agent scope (written through),
        // so waiting for our own stores is all the release there is - no write-back of the whole L2 - then take a ticket.
        unsigned ticket = 0;
        count_chunk<KMAX, false>(p, int(blockIdx.x), num_chunks, bitmap, nullptr, [&] {
            wait_for_own_stores();
            __syncthreads();
            if (tid == 0) ticket = atomicAdd(p.done_counter, 1u);
        });
        if (tid == 0) is_last = (ticket == unsigned(num_chunks) - 1u) ? 1 : 0;
        __syncthreads();
        if (!is_last) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");

        // ---- last workgroup: per-bucket totals, the public prefix sums and the row bases (LDS is re-carved) ----
        int* lds = reinterpret_cast<int*>(bitmap);
        if constexpr (kExpertsPerThread == 0) publish_layout<kThreads>(p.pub, p.tab, num_chunks, p.expert_bases != 0, lds);
        else publish_layout_in_one_trip<kThreads, false, kExpertsPerThread>(p.pub, p.tab, num_chunks, p.expert_bases != 0, nullptr, lds);
        if (tid == 0) *p.done_counter = 0u;                // ready for the next launch
    }
}

template <int KMAX>
void launch_layout(const LayoutParams& q, const IntranodePrefixParams& prefix, dim3 grid, size_t lds, bool one_chunk, hipStream_t stream) {
    const bool by_one = fits_one_trip(1, q.R, q.E, q.tab.chunks_padded, kThreads), by_two = fits_one_trip(2, q.R, q.E, q.tab.chunks_padded, kThreads);
    auto kernel = one_chunk ? (by_one ? layout_kernel<KMAX, true, 1> : layout_kernel<KMAX, true, 2>)
                : by_one    ? layout_kernel<KMAX, false, 1>
                : by_two    ? layout_kernel<KMAX, false, 2>
                            : layout_kernel<KMAX, false, 0>;
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), lds, stream, q, prefix);
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
    // LDS holds the bitmap words [R + E][kWaves] first; the last workgroup re-carves it for the publishing step, and the
    // only workgroup of a one-chunk call has its totals and the publishing step's scratch behind them.
    const size_t bitmap_bytes = count_lds_bytes(p.R, p.E);
    const size_t publish_bytes = publish_lds_bytes(p.R, p.E, kThreads);
    const size_t behind = (size_t(p.R + p.E) + publish_scratch_ints(p.R, kThreads)) * sizeof(int);
    const bool one_chunk = num_chunks == 1 && p.R <= kThreads && fits_one_trip(2, p.R, p.E, p.tab.chunks_padded, kThreads);
    size_t lds = one_chunk ? bitmap_bytes + behind : bitmap_bytes > publish_bytes ? bitmap_bytes : publish_bytes;
    if (prefix.R != 0 && lds < size_t(prefix.C) * sizeof(int)) lds = size_t(prefix.C) * sizeof(int);
    LayoutParams q = p;
    q.vec_idx = (reinterpret_cast<uintptr_t>(p.topk_idx) % 16 == 0) ? 1 : 0;
    const dim3 grid(num_chunks + prefix.R);
    if (p.K <= 8) launch_layout<8>(q, prefix, grid, lds, one_chunk, stream);
    else if (p.K <= 12) launch_layout<12>(q, prefix, grid, lds, one_chunk, stream);
    else if (p.K <= 16) launch_layout<16>(q, prefix, grid, lds, one_chunk, stream);
    else launch_layout<32>(q, prefix, grid, lds, one_chunk, stream);
    return hipGetLastError();
}

}  // namespace deep_ep_hip
