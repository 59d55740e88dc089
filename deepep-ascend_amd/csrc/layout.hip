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

// Bound by a chain of trips to memory, not by bytes: index loads, totals out, ticket, totals back, outputs.  Only the
// totals (and the flags) are waited for before the ticket; positions and copies are stored while it is on its way.  A
// call of one chunk hands its totals over in LDS instead.  Launch time, mailbox included, with everything
// waited for before the ticket and everything read back -> now: 128 tokens top-2 9.6 -> 6.1 us, 1237 top-9 13.0 -> 9.8,
// 4096 top-8 10.0 -> 8.3, 16384 top-8 over 32 ranks 14.8 -> 11.5.
template <int KMAX, bool kOneChunk>
__global__ __launch_bounds__(kThreads) void layout_kernel(const LayoutParams p) {
    extern __shared__ uint64_t bitmap[];   // [(R + E)][kWaves]
    __shared__ int is_last;
    const int tid = threadIdx.x;
    if constexpr (kOneChunk) {
        int* totals = reinterpret_cast<int*>(bitmap) + count_lds_bytes(p.R, p.E) / sizeof(int);
        count_chunk<KMAX, false>(p, 0, 1, bitmap, totals, [&] {
            wait_for_own_stores();                         // flags ORed into the status word, if any
            __syncthreads();
            publish_layout_in_one_trip<kThreads, true>(p.pub, p.tab, 1, p.expert_bases != 0, totals, totals + p.R + p.E);
        });
    } else {
        // Hand the chunk totals to whichever workgroup finishes last: they were stored at agent scope (written through),
        // so waiting for our own stores is all the release there is - no write-back of the whole L2 - then take a ticket.
        unsigned ticket = 0;
        count_chunk<KMAX, false>(p, int(blockIdx.x), int(gridDim.x), bitmap, nullptr, [&] {
            wait_for_own_stores();
            __syncthreads();
            if (tid == 0) ticket = atomicAdd(p.done_counter, 1u);
        });
        if (tid == 0) is_last = (ticket == gridDim.x - 1) ? 1 : 0;
        __syncthreads();
        if (!is_last) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");

        // ---- last workgroup: per-bucket totals, the public prefix sums and the row bases (LDS is re-carved) ----
        publish_layout<kThreads>(p.pub, p.tab, int(gridDim.x), p.expert_bases != 0, reinterpret_cast<int*>(bitmap));
        if (tid == 0) *p.done_counter = 0u;                // ready for the next launch
    }
}

template <int KMAX>
void launch_layout(const LayoutParams& q, dim3 grid, size_t lds, bool one_chunk, hipStream_t stream) {
    if (one_chunk) hipLaunchKernelGGL((layout_kernel<KMAX, true>), grid, dim3(kThreads), lds, stream, q);
    else hipLaunchKernelGGL((layout_kernel<KMAX, false>), grid, dim3(kThreads), lds, stream, q);
}

}  // namespace

hipError_t launch_layout_kernel(const LayoutParams& p, hipStream_t stream) {
    const int num_chunks = p.T > 0 ? (p.T + kThreads - 1) / kThreads : 1;
    // LDS holds the bitmap words [R + E][kWaves] first; the last workgroup re-carves it for the publishing step, and the
    // only workgroup of a one-chunk call has its totals and the publishing step's scratch behind them.
    const size_t bitmap_bytes = count_lds_bytes(p.R, p.E);
    const size_t publish_bytes = publish_lds_bytes(p.R, p.E, kThreads);
    const size_t behind = (size_t(p.R + p.E) + publish_scratch_ints(p.R, kThreads)) * sizeof(int);
    const bool one_chunk = num_chunks == 1 && p.R <= kThreads && p.E <= kThreads;
    const size_t lds = one_chunk ? bitmap_bytes + behind : bitmap_bytes > publish_bytes ? bitmap_bytes : publish_bytes;
    LayoutParams q = p;
    q.vec_idx = (reinterpret_cast<uintptr_t>(p.topk_idx) % 16 == 0) ? 1 : 0;
    const dim3 grid(num_chunks);
    if (p.K <= 8) launch_layout<8>(q, grid, lds, one_chunk, stream);
    else if (p.K <= 12) launch_layout<12>(q, grid, lds, one_chunk, stream);
    else if (p.K <= 16) launch_layout<16>(q, grid, lds, one_chunk, stream);
    else launch_layout<32>(q, grid, lds, one_chunk, stream);
    return hipGetLastError();
}

}  // namespace deep_ep_hip
