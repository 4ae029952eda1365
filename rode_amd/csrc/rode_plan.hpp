// The work of a workgroup that makes the descriptor of one chunk of a locality plan (rode_plan.hip), for the kernel that has the residue list
// and for the one that makes list and plan at once (rode_preprocess.hip).
#pragma once
#include "rode_items.hpp"

#include <climits>

namespace rode {

__device__ __forceinline__ int wave_reduce_add(int v)
{
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, kWave);
    return v;
}
__device__ __forceinline__ int wave_reduce_min(int v)
{
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v = min(v, __shfl_xor(v, d, kWave));
    return v;
}
__device__ __forceinline__ int wave_reduce_max(int v)
{
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) v = max(v, __shfl_xor(v, d, kWave));
    return v;
}

struct PlanChunkLds {
    int first[kPlanResidueChunk]; // first slot of every entry
    int prefix[kPlanResidueChunk + 1];
    __attribute__((aligned(16))) int samples[kWgThreads];
    int quart[2];
    int red[3][kWavesPerWg];
};

// The chunk whose entries start at the slots lds.first; my_len: slots of entry threadIdx.x (0 past the last).  Thread 0 returns the descriptor
// (first window row, rows, slots, slots outside).
__device__ __forceinline__ int4 plan_chunk(PlanChunkLds& lds, int my_len, int dense_rows, const int* __restrict__ col)
{
    constexpr int CH = kPlanResidueChunk;
    constexpr int ROWS_MAX = kResidueWindowRowsMax;
    static_assert(CH <= kWgThreads, "one thread per entry");
    int (&first)[CH] = lds.first;
    int (&prefix)[CH + 1] = lds.prefix;
    int (&samples)[kWgThreads] = lds.samples;
    int (&quart)[2] = lds.quart;
    int (&red)[3][kWavesPerWg] = lds.red;
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    static_assert(CH == 2 * kWave, "two waves have the entries");
    int through = my_len;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int up = __shfl_up(through, d, kWave);
        if (lane >= d) through += up;
    }
    if (tid == kWave - 1) red[0][0] = through;
    __syncthreads();
    if (tid < CH) prefix[tid + 1] = through + (wave > 0 ? red[0][0] : 0);
    if (tid == 0) prefix[0] = 0;
    if (tid < 2) quart[tid] = INT_MIN;
    __syncthreads();
    const int total = prefix[CH];
    if (total <= 0) {
        return make_int4(0, 0, 0, 0);
    }
    // entry that holds slot p of the chunk: the last e with prefix[e] <= p
    auto entry_of = [&](int p) {
        int lo = 0;
#pragma unroll
        for (int half = CH / 2; half > 0; half /= 2) lo += prefix[lo + half] <= p ? half : 0;
        return lo;
    };

    // 2. samples and their quartiles
    {
        const int p = (int)(((long long)tid * total + total / 2) / kWgThreads);
        const int e = entry_of(p);
        samples[tid] = col[first[e] + (p - prefix[e])];
    }
    __syncthreads();
    // the value of rank r is the largest one that at most r of the samples are below
    {
        const int mine = samples[tid];
        int below = 0;
#pragma unroll 4
        for (int j = 0; j < kWgThreads; j += 4) {
            const int4 other = *reinterpret_cast<const int4*>(samples + j);
            below += (other.x < mine ? 1 : 0) + (other.y < mine ? 1 : 0) + (other.z < mine ? 1 : 0) + (other.w < mine ? 1 : 0);
        }
        if (below <= kWgThreads / 4) atomicMax(quart, mine);
        if (below <= kWgThreads * 3 / 4 - 1) atomicMax(quart + 1, mine);
    }
    __syncthreads();
    const int q25 = quart[0], q75 = quart[1];
    if ((long long)q75 - q25 + 1 > ROWS_MAX || dense_rows <= 0) {
        return make_int4(0, 0, total, total);
    }
    int w0 = q25 + (q75 - q25) / 2 - ROWS_MAX / 2;
    w0 = max(0, min(w0, dense_rows - ROWS_MAX));
    const int wend = min(dense_rows, w0 + ROWS_MAX);

    // 3. hits and their extent
    int hits = 0, lo_hit = 0x7fffffff, hi_hit = -1;
    // (kAhead slots of a thread at a time: each is a search and a load that waits for it)
    constexpr int kAhead = 8;
    for (int p0 = tid; p0 < total; p0 += kAhead * kWgThreads) {
        int c[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int p = min(p0 + i * kWgThreads, total - 1), e = entry_of(p);
            c[i] = col[first[e] + (p - prefix[e])];
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (p0 + i * kWgThreads < total && c[i] >= w0 && c[i] < wend) {
                ++hits;
                lo_hit = min(lo_hit, c[i]);
                hi_hit = max(hi_hit, c[i]);
            }
        }
    }
    hits = wave_reduce_add(hits);
    lo_hit = wave_reduce_min(lo_hit);
    hi_hit = wave_reduce_max(hi_hit);
    if (lane == 0) {
        red[0][wave] = hits;
        red[1][wave] = lo_hit;
        red[2][wave] = hi_hit;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < kWavesPerWg; ++w) {
            hits += red[0][w];
            lo_hit = min(lo_hit, red[1][w]);
            hi_hit = max(hi_hit, red[2][w]);
        }
        // 4. decision
        const int wn = hi_hit - lo_hit + 1;
        const bool take = hits > 0 && 2ll * hits >= total && hits >= 2ll * wn;
        return make_int4(take ? lo_hit : 0, take ? wn : 0, total, total - hits);
    }
    return make_int4(0, 0, 0, 0);
}

} // namespace rode
