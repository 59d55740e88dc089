// Turning per-chunk totals into the public outputs of the layout computation (per-rank and per-expert counts,
// their prefix sums - the handle tensors of dispatch - and the host mailbox) and into the base tables the move
// kernels place rows with (struct LayoutTables).  Publishes what the notify warps of
// deep_ep/include/deep_ep/impls/dispatch.cuh:200-257 publish.
#pragma once

#include <type_traits>

#include "device_utils.h"
#include "kernels.h"

namespace deep_ep_hip {

// In-place inclusive scan of a[0..n) in LDS by the whole workgroup.  tmp holds one int per wavefront.
template <int kThreads>
__device__ void block_inclusive_scan(int* a, int n, int* tmp) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int per = (n + kThreads - 1) / kThreads;
    const int begin = min(tid * per, n), end = min(begin + per, n);
    int s = 0;
    for (int i = begin; i < end; ++i) s += a[i];
    const int inc = wave_inclusive_sum(s);
    if (lane == kWaveSize - 1) tmp[wave] = inc;
    __syncthreads();
    int run = inc - s;
    for (int w = 0; w < wave; ++w) run += tmp[w];
    for (int i = begin; i < end; ++i) {
        run += a[i];
        a[i] = run;
    }
    __syncthreads();
}

// LDS of the publishing workgroup: totals[R + E] | aligned[E] | aligned_incl[E] | one int per wavefront.
struct PublishLds {
    int* totals;         // rank part becomes its inclusive prefix sum in publish_ranks
    int* aligned;
    int* aligned_incl;
    int* scan_tmp;
};

__device__ __forceinline__ PublishLds carve_publish_lds(int* lds, int R, int E) {
    return PublishLds{lds, lds + R + E, lds + R + 2 * E, lds + R + 3 * E};
}

inline size_t publish_lds_bytes(int R, int E, int threads) {
    return size_t(R + 3 * E + threads / kWaveSize) * sizeof(int);
}

// ---- rank part: tables are transposed, [rank][chunk] ----

// totals[r] = sum of row r of rank_counts (padding columns are zero).  Ends with a barrier.
template <int kThreads>
__device__ void sum_rank_rows(const LayoutTables& t, int R, int* totals) {
    for (int j = threadIdx.x; j < R; j += kThreads) {
        const int32_t* row = t.rank_counts + int64_t(j) * t.chunks_padded;
        int sum = 0;
        for (int c0 = 0; c0 < t.chunks_padded; c0 += 32) {
            vec16 v[8];                                   // all loads of a pass in flight together
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = load16(row + min(c0 + 4 * u, t.chunks_padded - 4));
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c0 + 4 * u < t.chunks_padded) sum += int(v[u].x) + int(v[u].y) + int(v[u].z) + int(v[u].w);
        }
        totals[j] = sum;
    }
    __syncthreads();
}

// Per-rank outputs; afterwards s.totals[0..R) holds the inclusive prefix sum.  Every thread must call it.
template <int kThreads>
__device__ void publish_ranks(const PublishParams& q, const PublishLds& s) {
    for (int r = threadIdx.x; r < q.R; r += kThreads) {
        if (q.num_tokens_per_rank != nullptr) q.num_tokens_per_rank[r] = s.totals[r];
        if (q.host_counts != nullptr) store_system(q.host_counts + r, -s.totals[r] - 1);
    }
    __syncthreads();
    block_inclusive_scan<kThreads>(s.totals, q.R, s.scan_tmp);
    for (int r = threadIdx.x; r < q.R; r += kThreads)
        if (q.psum_rank != nullptr) q.psum_rank[r] = s.totals[r];
    if (threadIdx.x == 0 && q.totals_out != nullptr) q.totals_out[0] = s.totals[q.R - 1];
}

// rank_bases[r][c] = (rows of lower ranks) + sum of rank_counts[r][0..c): one thread per rank, 32 chunks per pass
// with all of a pass's loads in flight together.  s.totals[0..R) must hold the inclusive prefix sum of the ranks.
template <int kThreads>
__device__ void write_rank_bases(const LayoutTables& t, int R, const PublishLds& s) {
    for (int j = threadIdx.x; j < R; j += kThreads) {
        const int32_t* src = t.rank_counts + int64_t(j) * t.chunks_padded;
        int32_t* dst = t.rank_bases + int64_t(j) * t.chunks_padded;
        int run = j > 0 ? s.totals[j - 1] : 0;
        for (int c0 = 0; c0 < t.chunks_padded; c0 += 32) {
            vec16 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = load16(src + min(c0 + 4 * u, t.chunks_padded - 4));
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (c0 + 4 * u < t.chunks_padded) {
                    vec16 o;
                    o.x = uint32_t(run); run += int(v[u].x);
                    o.y = uint32_t(run); run += int(v[u].y);
                    o.z = uint32_t(run); run += int(v[u].z);
                    o.w = uint32_t(run); run += int(v[u].w);
                    store16(dst + c0 + 4 * u, o);
                }
            }
        }
    }
}

// The rank part as one flat pass over rank_counts ([rank][chunk], R * chunks_padded <= 4 * kThreads entries), for the
// publishing workgroup of a single-launch dispatch.  A line of that table holds the totals of up to 16 chunks, written
// through by as many counting workgroups of the same launch, some of them on this XCD: it is read at agent scope, past
// any partial copy of the line a cache may hold.  The inclusive prefix sum over the flattened table is, at the last
// entry of row r, the end of rank r's bucket.  Publishes the per-rank outputs.  Every thread of the workgroup must
// call it; s.scan_tmp: kThreads / 64 ints of LDS.
template <int kThreads>
__device__ void scan_rank_counts(const PublishParams& q, const LayoutTables& t, int R, const PublishLds& s) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int flat = R * t.chunks_padded;              // a multiple of 4: a thread's entries share a row
    const int begin = tid * 4;
    vec16 v{0, 0, 0, 0};
    if (begin < flat) {
        const unsigned long long* at = reinterpret_cast<const unsigned long long*>(t.rank_counts + begin);
        const unsigned long long lo = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long hi = __hip_atomic_load(at + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        v = vec16{uint32_t(lo), uint32_t(lo >> 32), uint32_t(hi), uint32_t(hi >> 32)};
    }
    const int sum = int(v.x) + int(v.y) + int(v.z) + int(v.w);
    const int inc = wave_inclusive_sum(sum);
    if (lane == kWaveSize - 1) s.scan_tmp[wave] = inc;
    __syncthreads();
    int run = inc - sum;
    for (int w = 0; w < wave; ++w) run += s.scan_tmp[w];
    if (begin < flat && (begin + 4) % t.chunks_padded == 0) s.totals[begin / t.chunks_padded] = run + sum;   // inclusive prefix of the rank
    __syncthreads();
    for (int r = tid; r < R; r += kThreads) {
        const int total = s.totals[r] - (r > 0 ? s.totals[r - 1] : 0);
        if (q.num_tokens_per_rank != nullptr) q.num_tokens_per_rank[r] = total;
        if (q.host_counts != nullptr) store_system(q.host_counts + r, -total - 1);
        if (q.psum_rank != nullptr) q.psum_rank[r] = s.totals[r];
    }
    if (tid == 0 && q.totals_out != nullptr) q.totals_out[0] = s.totals[R - 1];
}

// ---- expert part: tables are [chunk][expert], so that thread e walks column e with coalesced accesses ----

// totals[R + e] = sum over chunks of expert_counts[c][e].  Ends with a barrier.
template <int kThreads>
__device__ void sum_expert_columns(const LayoutTables& t, int R, int E, int num_chunks, int* totals) {
    for (int e = threadIdx.x; e < E; e += kThreads) {
        const int32_t* col = t.expert_counts + e;
        int sum = 0;
        for (int c0 = 0; c0 < num_chunks; c0 += 16) {
            int v[16];                                    // all loads of a pass in flight together
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = col[int64_t(min(c0 + u, num_chunks - 1)) * t.experts_padded];
#pragma unroll
            for (int u = 0; u < 16; ++u) sum += c0 + u < num_chunks ? v[u] : 0;
        }
        totals[R + e] = sum;
    }
    __syncthreads();
}

// First thread: the status word as the counting workgroups left it (they are all done when a workgroup publishes), for
// the host's mailbox.  Asked for early: the trip to memory passes beside the prefix sums.
__device__ __forceinline__ int status_for_host(const PublishParams& q) {
    return threadIdx.x == 0 && q.host_counts != nullptr && q.status != nullptr ? load_agent(q.status) : 0;
}

// Per-expert outputs; afterwards the region of expert j starts at s.aligned_incl[j] - s.aligned[j].
//
// The words of the mailbox are stored at system scope, each valid by itself (v as -v-1): the host sees a word as soon as
// it has crossed the bus, and no fence follows.  With a system-scope fence, which writes the whole L2 back and waits for
// it, a layout launch took 1 to 2 us longer.
template <int kThreads>
__device__ void publish_experts(const PublishParams& q, const PublishLds& s, const int status) {
    for (int j = threadIdx.x; j < q.E; j += kThreads) {
        const int cnt = s.totals[q.R + j];
        const int al = (cnt + q.A - 1) / q.A * q.A;
        s.aligned[j] = al;
        s.aligned_incl[j] = al;
        if (q.num_tokens_per_expert != nullptr) q.num_tokens_per_expert[j] = cnt;
        if (q.num_unaligned != nullptr) q.num_unaligned[j] = cnt;
        if (q.cumulative_stats != nullptr) q.cumulative_stats[j] += cnt;
        if (q.host_counts != nullptr) store_system(q.host_counts + q.R + j, -al - 1);
    }
    __syncthreads();
    block_inclusive_scan<kThreads>(s.aligned_incl, q.E, s.scan_tmp);
    for (int j = threadIdx.x; j < q.E; j += kThreads) {
        const int start = s.aligned_incl[j] - s.aligned[j];
        if (q.expert_start != nullptr) q.expert_start[j] = start;
        if (q.psum_expert != nullptr) q.psum_expert[j] = q.do_expand ? start + s.totals[q.R + j] : s.aligned_incl[j];
    }
    if (threadIdx.x == 0 && q.totals_out != nullptr) q.totals_out[1] = q.E > 0 ? s.aligned_incl[q.E - 1] : 0;
    // The status word: a host that sizes its outputs from this mailbox learns about bad routing input without a second
    // trip to the device.
    if (threadIdx.x == 0 && q.host_counts != nullptr) store_system(q.host_counts + q.R + q.E, -status - 1);
}

// table[c][e] = start of expert e's region + sum of expert_counts[0..c)[e], each word ORed with `tag`.
// kThrough: stored at agent scope.
template <int kThreads, bool kThrough>
__device__ void write_expert_bases(const LayoutTables& t, int32_t* table, uint32_t tag, int E, int num_chunks, const PublishLds& s) {
    for (int e = threadIdx.x; e < E; e += kThreads) {
        const int32_t* col = t.expert_counts + e;
        int32_t* out = table + e;
        int run = s.aligned_incl[e] - s.aligned[e];
        for (int c0 = 0; c0 < num_chunks; c0 += 16) {
            int v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = col[int64_t(min(c0 + u, num_chunks - 1)) * t.experts_padded];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                if (c0 + u < num_chunks) {
                    store_word<kThrough>(out + int64_t(c0 + u) * t.experts_padded, int(uint32_t(run) | tag));
                    run += v[u];
                }
            }
        }
    }
}

// Does `word` carry the tag of the running single-launch dispatch (kernels.h)?
__device__ __forceinline__ bool has_tag(uint32_t word, uint32_t tag) {
    return (word & ~kTagValueMask) == tag;
}

// The expert base table in one trip, for the publishing workgroup of a single-launch expanded dispatch, whose movers
// wait for exactly this.  Thread e reads its column of the tagged chunk totals at agent scope, again (at most
// spin_limit times) until every word shows the tag - no flag of the counting workgroups is waited for, which would
// only be raised once all their stores are acknowledged - keeps the column in registers between the sum and the
// stores, and stores the bases at agent scope, each ORed with `tag`.  Needs E <= kThreads and num_chunks <= 32.
// Leaves totals / aligned / aligned_incl as publish_experts expects to recompute them.  A: expert alignment.
// Returns whether every thread got its column.
template <int kThreads>
__device__ bool write_expert_bases_from_registers(const LayoutTables& t, const uint32_t* tagged_counts, int32_t* table, uint32_t tag,
                                                  unsigned spin_limit, int R, int E, int A, int num_chunks, const PublishLds& s) {
    const int e = threadIdx.x;
    int v[32];
    int total = 0;
    bool complete = true;
    if (e < E) {
        unsigned polls = 0;
        for (;;) {
            complete = true;
#pragma unroll
            for (int u = 0; u < 32; ++u) {
                // a row start common to the workgroup plus the thread's column: one address register serves all 32 loads
                const int row_start = __builtin_amdgcn_readfirstlane(min(u, num_chunks - 1) * t.experts_padded);
                v[u] = load_agent(reinterpret_cast<const int*>(tagged_counts) + row_start + e);
            }
#pragma unroll
            for (int u = 0; u < 32; ++u) complete = complete && has_tag(uint32_t(v[u]), tag);
            if (complete || polls == spin_limit) break;
            __builtin_amdgcn_s_sleep(4);
            ++polls;
        }
#pragma unroll
        for (int u = 0; u < 32; ++u) {
            v[u] = int(uint32_t(v[u]) & kTagValueMask);
            total += u < num_chunks ? v[u] : 0;
        }
        s.totals[R + e] = total;
        const int al = (total + A - 1) / A * A;
        s.aligned[e] = al;
        s.aligned_incl[e] = al;
    }
    const int all_complete = __syncthreads_and(complete ? 1 : 0);
    block_inclusive_scan<kThreads>(s.aligned_incl, E, s.scan_tmp);
    if (e < E) {
        int run = s.aligned_incl[e] - s.aligned[e];
#pragma unroll
        for (int u = 0; u < 32; ++u) {
            if (u < num_chunks) {
                const int row_start = __builtin_amdgcn_readfirstlane(u * t.experts_padded);
                store_agent(table + row_start + e, int(uint32_t(run) | tag));
                run += v[u];
            }
        }
    }
    return all_complete != 0;
}

// publish_layout for the common sizes: num_experts <= kPerThread * kThreads, R * chunks_padded <= 16 * kThreads (fits_one_trip).  A workgroup of its
// own on the critical path of every call: what it costs is the chain of barriers, LDS trips and instruction fetches, so
// there is one trip to memory (every thread first loads all it needs: up to 16 consecutive entries of the flattened rank
// table and its experts' columns of chunk totals, of which 32 stay in registers), one pair of prefix sums, taken
// together, and two barriers; outputs go out from registers.  kHeldChunks > 0: `totals` ([R + E][kHeldChunks], LDS) holds all
// chunks' totals and nothing is loaded.  scratch: LDS of publish_scratch_ints.
// From the ticket to the end it took 3.4 us at 16 chunks, 9 us at 64 chunks over 32 ranks, with LDS scans of five
// barriers and 32 chunks at most; the whole launch went from 10.0 to 8.3 and from 14.8 to 11.5 us.
// Chunks past the 32 in registers are read again for the expert bases, sixteen a trip: one at a time, each load behind the store
// before it, an expanded layout took 41.7 us at 65536 tokens over 8 ranks, 13.8 at 16384 over 32, and takes 29.1 and 12.2.
// Two experts a thread: the layout launch over 512 experts of 16 ranks took 11.8 us at 57 tokens, 13.3 at 8192 (expanded 16.6) and 18.0 at
// 20000 (26.0) in the steps of publish_layout, and takes 7.0, 9.3 (10.8) and 11.5 (16.2).  A launch's kernel holds only its own way of
// publishing: with the two-expert one beside it the launch took 0.2 to 0.4 us longer over 256 experts.
inline bool fits_one_trip(int per_thread, int R, int E, int chunks_padded, int threads) {
    return E <= per_thread * threads && R * chunks_padded <= 16 * threads;
}

inline __host__ __device__ int publish_scratch_ints(int R, int threads) { return R + 2 * (threads / kWaveSize); }

template <int kThreads, int kHeldChunks, int kPerThread>
__device__ void publish_layout_in_one_trip(const PublishParams& q, const LayoutTables& t, int num_chunks, bool expert_bases,
                                           int* totals, int* scratch) {
    constexpr int kWavesHere = kThreads / kWaveSize;
    static_assert(kHeldChunks <= 4 && (kPerThread == 1 || kHeldChunks <= 1), "rows of four chunks; for_host lies over the totals");
    constexpr bool kHeld = kHeldChunks > 0;
    constexpr int kMaxVecs = kHeld ? 1 : 4, kColumn = kHeld ? kHeldChunks : 32 / kPerThread;
    int* rank_end = scratch;                             // [R] inclusive prefix sum over the ranks
    int* wave_sums = scratch + q.R;                      // [2][kWavesHere]
    // kPerThread > 1: [E] what the mailbox gets, of which a thread writes the entries it has read the totals from
    int* for_host = kHeld ? totals + q.R : scratch + publish_scratch_ints(q.R, kThreads);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int first_expert = tid * kPerThread;
    const bool has_expert = first_expert < q.E;
    const int status = status_for_host(q);
    const int flat = q.R * t.chunks_padded;              // a multiple of 4: four entries share a row
    const int vecs = kHeld ? 1 : (flat + 4 * kThreads - 1) / (4 * kThreads);
    // The thread's experts of a chunk: columns the table pads with (experts_padded is a multiple of 32) come along and count nothing.
    // Tables are read and written through descriptors that end with them: chunks there are none of count zero and are not stored, with no
    // test and no address for each (a wavefront here has its SIMD to itself: every instruction counts).
    using Columns = std::conditional_t<kPerThread == 1, uint32_t, uint2>;
    const auto of = [](auto& columns, int j) -> uint32_t& { return reinterpret_cast<uint32_t*>(&columns)[j]; };
    const uint32_t row_bytes = uint32_t(t.experts_padded) * 4u, my_columns = uint32_t(has_expert ? first_expert : 0) * 4u;
    const auto expert_counts = buffer_of(reinterpret_cast<const uint8_t*>(t.expert_counts), kHeld ? 0 : num_chunks * int(row_bytes));
    vec16 rv[kMaxVecs];
    Columns v[kColumn];
    int rows = 0, count[kPerThread] = {};
    auto load_rows = [&](int first, auto& to, int from, int n) {
        uint32_t at = uint32_t(first) * row_bytes + my_columns;
#pragma unroll
        for (int u = 0; u < 16; ++u, at += row_bytes)
            if (u < n) to[from + u] = buffer_load_words<Columns>(expert_counts, at);
    };
    if constexpr (kHeld) {
        const auto total = [&](int bucket, int chunk, bool there) { return there && chunk < kHeldChunks ? totals[bucket * kHeldChunks + min(chunk, kHeldChunks - 1)] : 0; };
        const bool has_rank = tid < q.R;                 // rows of four, some of them padding
        rv[0] = vec16{uint32_t(total(tid, 0, has_rank)), uint32_t(total(tid, 1, has_rank)), uint32_t(total(tid, 2, has_rank)), uint32_t(total(tid, 3, has_rank))};
#pragma unroll
        for (int c = 0; c < kHeldChunks; ++c)
#pragma unroll
            for (int j = 0; j < kPerThread; ++j) {
                of(v[c], j) = uint32_t(total(q.R + first_expert + j, c, first_expert + j < q.E));
                count[j] += int(of(v[c], j));
            }
        rows = int(rv[0].x) + int(rv[0].y) + int(rv[0].z) + int(rv[0].w);
    } else {
        const auto rank_counts = buffer_of(reinterpret_cast<const uint8_t*>(t.rank_counts), flat * 4);
#pragma unroll
        for (int i = 0; i < kMaxVecs; ++i) {
            rv[i] = vec16{0, 0, 0, 0};
            if (i < vecs) rv[i] = buffer_load16_as<false>(rank_counts, (tid * vecs + i) * 16);
        }
        auto sum_rows = [&](auto& of_chunks, int n) {
#pragma unroll
            for (int u = 0; u < n; ++u)
#pragma unroll
                for (int j = 0; j < kPerThread; ++j) count[j] += int(of(of_chunks[u], j));
        };
#pragma unroll
        for (int c0 = 0; c0 < kColumn; c0 += 8) {
            if (c0 < num_chunks) {
                load_rows(c0, v, c0, 8);
            } else {
#pragma unroll
                for (int u = 0; u < 8; ++u) v[c0 + u] = Columns{};
            }
        }
        for (int c0 = kColumn; c0 < num_chunks; c0 += 16) {
            Columns w[16];
            load_rows(c0, w, 0, 16);
            sum_rows(w, 16);
        }
        sum_rows(v, kColumn);
#pragma unroll
        for (int i = 0; i < kMaxVecs; ++i) rows += int(rv[i].x) + int(rv[i].y) + int(rv[i].z) + int(rv[i].w);
    }
    int aligned[kPerThread], all_aligned = 0;
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        aligned[j] = 0;
        if (first_expert + j < q.E) aligned[j] = q.A == 1 ? count[j] : int((unsigned(count[j]) + unsigned(q.A) - 1u) / unsigned(q.A)) * q.A;
        all_aligned += aligned[j];
    }

    const int rows_incl = wave_inclusive_sum(rows), aligned_incl = wave_inclusive_sum(all_aligned);
    if (lane == kWaveSize - 1) {
        wave_sums[wave] = rows_incl;
        wave_sums[kWavesHere + wave] = aligned_incl;
    }
    __syncthreads();
    int run = rows_incl - rows, start = aligned_incl - all_aligned;
#pragma unroll
    for (int w = 0; w < kWavesHere - 1; ++w) {
        run += w < wave ? wave_sums[w] : 0;
        start += w < wave ? wave_sums[kWavesHere + w] : 0;
    }
    Columns base;                                        // the region of an expert starts at the aligned rows of those before it
#pragma unroll
    for (int j = 0, at = start; j < kPerThread; at += aligned[j], ++j) of(base, j) = uint32_t(at);

#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        const int e = first_expert + j;
        if (e >= q.E) break;
        if constexpr (kPerThread > 1) for_host[e] = aligned[j];
        else if (q.host_counts != nullptr) store_system(q.host_counts + q.R + e, -aligned[j] - 1);
        if (q.num_tokens_per_expert != nullptr) q.num_tokens_per_expert[e] = count[j];
        if (q.num_unaligned != nullptr) q.num_unaligned[e] = count[j];
        if (q.cumulative_stats != nullptr) q.cumulative_stats[e] += count[j];
        if (q.expert_start != nullptr) q.expert_start[e] = int(of(base, j));
        if (q.psum_expert != nullptr) q.psum_expert[e] = q.do_expand ? int(of(base, j)) + count[j] : int(of(base, j)) + aligned[j];
        if (e == q.E - 1 && q.totals_out != nullptr) q.totals_out[1] = int(of(base, j)) + aligned[j];
    }
    // ranks: the exclusive prefix over the flattened table is the first compact row of every (rank, chunk)
    const float rcp_row = 1.0f / float(t.chunks_padded);
#pragma unroll
    for (int i = 0; i < kMaxVecs; ++i) {
        const int begin = (tid * vecs + i) * 4;
        if (i >= vecs || begin >= flat) break;
        const uint32_t b0 = uint32_t(run), b1 = b0 + rv[i].x, b2 = b1 + rv[i].y, b3 = b2 + rv[i].z;
        run = int(b3 + rv[i].w);
        if (t.rank_bases != nullptr) store16(t.rank_bases + begin, vec16{b0, b1, b2, b3});
        const int r = small_div(begin, rcp_row);
        if (begin + 4 == (r + 1) * t.chunks_padded) rank_end[r] = run;
    }
    __syncthreads();
    // Neighbouring lanes store neighbouring words: every second word at a time the bus takes them one by one, which kept the host
    // waiting 45 us longer over 512 experts.
    if constexpr (kPerThread > 1)
        if (q.host_counts != nullptr)
            for (int e = tid; e < q.E; e += kThreads) store_system(q.host_counts + q.R + e, -for_host[e] - 1);
    for (int r = tid; r < q.R; r += kThreads) {
        const int end = rank_end[r], total = end - (r > 0 ? rank_end[r - 1] : 0);
        if (q.host_counts != nullptr) store_system(q.host_counts + r, -total - 1);
        if (q.num_tokens_per_rank != nullptr) q.num_tokens_per_rank[r] = total;
        if (q.psum_rank != nullptr) q.psum_rank[r] = end;
        if (r == q.R - 1 && q.totals_out != nullptr) q.totals_out[0] = end;
    }
    if (tid == 0 && q.host_counts != nullptr) store_system(q.host_counts + q.R + q.E, -status - 1);

    if (t.expert_bases != nullptr && expert_bases && has_expert) {
        const auto table = buffer_of(reinterpret_cast<const uint8_t*>(t.expert_bases), num_chunks * int(row_bytes));
        uint32_t at = my_columns;
        auto store_base = [&](Columns& counts) {
            buffer_store_words(table, at, base);
            at += row_bytes;
#pragma unroll
            for (int j = 0; j < kPerThread; ++j) of(base, j) += of(counts, j);
        };
        if constexpr (kHeld) {
#pragma unroll
            for (int u = 0; u < kColumn; ++u) store_base(v[u]);
        } else {
#pragma unroll
            for (int c0 = 0; c0 < kColumn; c0 += 8) {
                if (c0 >= num_chunks) break;
#pragma unroll
                for (int u = 0; u < 8; ++u) store_base(v[c0 + u]);
            }
            for (int c0 = kColumn; c0 < num_chunks; c0 += 16) {
                Columns w[16];
                load_rows(c0, w, 0, 16);
#pragma unroll
                for (int u = 0; u < 16; ++u) store_base(w[u]);
            }
        }
    }
}

// Everything at once, for a workgroup that publishes after all counting is over (the stand-alone layout kernel):
// totals, public outputs, and - when the caller has room for them - the base tables.  Any sizes.
template <int kThreads>
__device__ void publish_layout(const PublishParams& q, const LayoutTables& t, int num_chunks, bool expert_bases, int* lds) {
    const PublishLds s = carve_publish_lds(lds, q.R, q.E);
    const int status = status_for_host(q);
    sum_rank_rows<kThreads>(t, q.R, s.totals);
    sum_expert_columns<kThreads>(t, q.R, q.E, num_chunks, s.totals);
    publish_ranks<kThreads>(q, s);
    __syncthreads();
    if (t.rank_bases != nullptr) write_rank_bases<kThreads>(t, q.R, s);
    publish_experts<kThreads>(q, s, status);
    if (t.expert_bases != nullptr && expert_bases) {
        __syncthreads();
        write_expert_bases<kThreads, false>(t, t.expert_bases, 0u, q.E, num_chunks, s);
    }
}

}  // namespace deep_ep_hip
