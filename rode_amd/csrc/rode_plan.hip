// Locality plan: for every chunk of 128 consecutive residue-list entries, decide whether
// the dense rows its nonzeros reference cluster in a window of consecutive rows small
// enough to be staged in LDS (banded matrices), and which window.
//
// No counterpart in the reference: its kernels gather every dense row from memory
// (RoDe_SpMM/RoDeSpmm.cu:140-160, RoDe_SDDMM/RoDeSddmm.cu:96-140).  The plan changes no
// result; it only tells the window kernels where most of a chunk's dense rows are.
//
// One workgroup per chunk:
//   1. slot range of every entry (the ranges of RoDeSpmm.cu:71-82);
//   2. 256 column samples spread evenly over the chunk's slots; their quartiles q25 and
//      q75 place the window: if they are further apart than the window is long, the chunk
//      has no window; otherwise the window is centred on their midpoint;
//   3. every slot is tested against that window: hit count and the extent of the hits
//      (the window shrinks to [smallest hit, largest hit]);
//   4. the chunk gets its window if the hits are at least half of its slots and at least
//      twice the window's rows (staging a row has to be repaid by about two reads).
//
// What bounds it: the chain of loads that wait for one another (list entry, row offset, column), with a few workgroups
// per CU; 65 K rows with 2 M nonzeros: 14.1 us with the counts written to the host from here, 15.5 with one slot of a thread
// at a time.  Before, 13.2, a launch of 2.0 that set up the header and a copy of 3.7 that brought the counts to the host.
#include "rode_plan.hpp"
#include "rode_internal.hpp"

namespace rode {

namespace {

__global__ void plan_header_kernel(int m2, int windowed, int* __restrict__ plan)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        plan[0] = plan_residue_chunks(m2);
        plan[1] = windowed;
        plan[2] = 0;
        plan[3] = 0;
    }
}

__global__ void __launch_bounds__(kWgThreads)
plan_chunks_kernel(int m2, int dense_rows, const int* __restrict__ residue_rows, const int* __restrict__ row_ptr,
                   const int* __restrict__ col, int* plan, int* host_counts)
{
    constexpr int CH = kPlanResidueChunk;
    __shared__ PlanChunkLds lds;
    const int tid = threadIdx.x;
    const int chunk = blockIdx.x;
    const int e0 = chunk * CH;
    const int ne = min(CH, m2 - e0);
    int* desc = plan + kPlanHeaderInts + kPlanDescInts * chunk;
    // (one thread) the chunk's descriptor; where the counts go to the host, the last chunk to come here writes them there (one
    // 64-bit counter in the header's last two ints, which end as zero: the chunks done, and above them those with a window)
    auto finish = [&](int4 d) {
        *reinterpret_cast<int4*>(desc) = d;
        const int wn = d.y;
        if (host_counts == nullptr) {
            if (wn > 0) atomicAdd(plan + 1, 1);
            return;
        }
        unsigned long long* counter = reinterpret_cast<unsigned long long*>(plan + 2);
        const unsigned long long mine = 1ull + (wn > 0 ? 1ull << 32 : 0ull);
        const unsigned long long all = atomicAdd(counter, mine) + mine;
        if ((unsigned)all != gridDim.x) return;
        const int windowed = (int)(all >> 32);
        plan[1] = windowed, *counter = 0;
        host_counts[0] = gridDim.x, host_counts[1] = windowed, host_counts[2] = 0, host_counts[3] = 0;
    };

    int my_len = 0;
    if (tid < ne) {
        const ResidueItem it = residue_item(residue_rows[e0 + tid], row_ptr);
        lds.first[tid] = it.first;
        my_len = it.cnt;
    }
    const int4 d = plan_chunk(lds, my_len, dense_rows, col);
    if (tid == 0) finish(d);
}

// Fills the PlannedChunk of every chunk that has a window: 8 threads per residue row.
__global__ void __launch_bounds__(kPlanResidueChunk * 8)
plan_rows_kernel(int m2, const int* __restrict__ residue_rows, const int* __restrict__ row_ptr,
                 const int* __restrict__ col, const int* __restrict__ plan, PlannedChunk* __restrict__ rows)
{
    constexpr int L = 8, OWN = kBlockItems / L;
    __shared__ unsigned char keys[kPlanResidueChunk][kBlockItems];
    const int chunk = blockIdx.x;
    const WindowDesc d = plan_residue_desc(plan, chunk);
    PlannedChunk& out = rows[chunk];
    if (threadIdx.x == 0) {
        out.w0 = d.w0;
        out.wn = d.wn;
        out.next = out.reserved = 0;
    }
    if (d.wn <= 0) {
        const int ahead = chunk + 1 + (int)threadIdx.x;
        if (threadIdx.x < kWave) {
            const unsigned long long windows = __ballot(ahead < (int)gridDim.x && plan_residue_desc(plan, min(ahead, (int)gridDim.x - 1)).wn > 0);
            if (threadIdx.x == 0) out.next = windows ? __builtin_ctzll(windows) + 1 : kWave + 1;
        }
        return;
    }
    const int local = threadIdx.x / L, ls = threadIdx.x % L;
    const int entry = chunk * kPlanResidueChunk + local;
    int row = -1, first = 0, cnt = 0, aligned = 0;
    bool accumulate = false;
    if (entry < m2) {
        row = residue_rows[entry];
        const ResidueItem it = residue_item(row, row_ptr);
        first = it.first;
        cnt = it.cnt;
        aligned = it.aligned;
        accumulate = it.accumulate;
    }
    // which lane group of the window kernels takes this row: groups 2, 3, 6, 7 list odd window rows first
    const int odd_first = (local >> 1) & 1;
    unsigned u[OWN];
    unsigned best = 0xffffu;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int s = ls + i * L;
        u[i] = 0xffffu;
        unsigned char key = 3; // not a slot of the row
        if (s < cnt) {
            const unsigned dw = (unsigned)(col[first + s] - d.w0);
            if (dw < (unsigned)d.wn) {
                u[i] = dw;
                key = ((dw & 1u) != (unsigned)odd_first) ? 1 : 0;
            } else {
                key = 2; // outside the window: after the ones inside
            }
        }
        keys[local][s] = key;
        best = min(best, u[i]);
    }
#pragma unroll
    for (int m = 1; m < L; m <<= 1) best = min(best, (unsigned)__shfl_xor((int)best, m, kWave));
    const bool none_inside = best == 0xffffu && cnt > 0;
    if (best == 0xffffu) best = 0; // no slot inside the window: every read is replaced, those of places that the row does not fill too (by
                                   // its first slot's: the window's first row is none of this row's, and may hold what times zero is not zero)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); // the 8 threads of a row are lanes of one wave
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    unsigned missbits = 0;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int s = ls + i * L;
        const int key = keys[local][s];
        int rank = 0; // position: slots with a smaller key, or the same key and a smaller index, come first
        for (int o = 0; o < kBlockItems; ++o) {
            const int other = keys[local][o];
            rank += (other < key || (other == key && o < s)) ? 1 : 0;
        }
        const unsigned where = key == 0 || key == 1 ? u[i] : best;
        out.entry[local][rank] = (unsigned short)(where | (key <= 2 ? (unsigned)s << 9 : 0u));
        if (key == 2 || none_inside) missbits |= 1u << rank;
    }
#pragma unroll
    for (int m = 1; m < L; m <<= 1) missbits |= (unsigned)__shfl_xor((int)missbits, m, kWave);
    if (ls == 0) {
        PlannedRowMeta meta;
        meta.row = row;
        meta.first = first;
        meta.packed = cnt | (accumulate ? 1 << 8 : 0) | (min(aligned, 0xffff) << 16);
        meta.missmask = missbits;
        out.meta[local] = meta;
    }
}

} // namespace

size_t window_plan_ints(int m2) { return plan_ints(m2); }
int window_plan_chunks(int m2) { return plan_residue_chunks(m2); }
size_t window_plan_rows_bytes(int m2) { return (size_t)plan_residue_chunks(m2) * sizeof(PlannedChunk); }

hipError_t window_plan_header_launch(int m2, int windowed, int* plan, hipStream_t stream)
{
    plan_header_kernel<<<1, kWave, 0, stream>>>(m2, windowed, plan);
    return hipGetLastError();
}

hipError_t window_plan_launch(int m2, int dense_rows, const int* residue_rows, const int* row_ptr, const int* col,
                              int* plan, hipStream_t stream, int* header_counts)
{
    if (header_counts == nullptr) plan_header_kernel<<<1, kWave, 0, stream>>>(m2, 0, plan);
    const int chunks = plan_residue_chunks(m2);
    if (chunks > 0) {
        plan_chunks_kernel<<<chunks, kWgThreads, 0, stream>>>(m2, dense_rows, residue_rows, row_ptr, col, plan, header_counts);
    }
    return hipGetLastError();
}

hipError_t window_plan_rows_launch(int m2, const int* residue_rows, const int* row_ptr, const int* col, const int* plan,
                                   void* rows, hipStream_t stream)
{
    const int chunks = plan_residue_chunks(m2);
    if (chunks > 0)
        plan_rows_kernel<<<chunks, kPlanResidueChunk * 8, 0, stream>>>(m2, residue_rows, row_ptr, col, plan,
                                                                       static_cast<PlannedChunk*>(rows));
    return hipGetLastError();
}

} // namespace rode
