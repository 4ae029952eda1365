// Pieces shared by the window kernels of SpMM and SDDMM (rode_spmm_window.hip,
// rode_sddmm_window.hip): the kernels for chunks of the residue list whose dense rows
// cluster in a window of consecutive rows (see the locality plan in rode_items.hpp).
//
// Shape of both kernels.  A workgroup of 1024 threads per CU walks chunks of the plan (128
// consecutive residue rows), one group of 8 lanes per row, and for each chunk the column tiles
// of 128 bytes (32 fp32, 64 fp16, 16 fp64 columns) of the dense operand.  Per tile the rows
// [w0, w0 + wn) of the operand - the chunk's window - are copied into LDS once, and every
// nonzero slot whose column falls into the window reads its dense row there (8 lanes x
// ds_read_b128, one contiguous 128-byte row per lane group) instead of gathering it from L2; a
// slot outside the window is gathered from memory.  Which window row a slot reads is not worked
// out here: the plan holds it for every residue row of a chunk with a window (PlannedChunk), in
// an order that keeps lane groups that meet in the LDS banks on rows of different parity.
//
// What bounds them: for 128 columns of fp32, memory (the operands once, 80 % of a large copy's
// rate) and the work on a tile (LDS reads and multiply-adds) take about as long as each other, so
// everything is there to have both going all the time.  The copies go from memory to LDS without
// registers in between, a tile ahead of the work (the next chunk's first tile during the last of
// this one, and its record during the first); two windows and two records fill the LDS of a CU, hence
// the one workgroup, which stays and takes chunk after chunk.  Measured on the banded benchmark
// (1 M rows, band of 256) against two workgroups of 512 threads per CU that each took half a chunk and
// loaded a tile between two barriers: SDDMM of width 128 0.531 -> 0.388 ms, width 64 0.361 -> 0.246, 500 K rows
// of 128 halves 0.217 -> 0.141.  Of the 0.388 the work alone would take 0.301 and the copies alone 0.304.
// Tried: LDS reads of the next four slots between the multiply-adds of these (0.465).
#pragma once
#include "rode_items.hpp"

#include <cstddef>

namespace rode {

constexpr int kResLanes = 8;                                   // lanes per residue row: 8 x 16 bytes = one 128-byte tile row
constexpr int kResThreads = kPlanResidueChunk * kResLanes;     // a workgroup takes a chunk
constexpr int kResWinVecs = kResidueWindowRowsMax * kResLanes; // 16-byte pieces of a window
constexpr int kRecordVecs = (int)sizeof(PlannedChunk) / 16;    // ... of a chunk's record
constexpr int kRecordRoom = (kRecordVecs + kWave - 1) / kWave * kWave; // (a wave copies 64 pieces, needed or not)
static_assert(kResThreads <= 1024, "a workgroup");
static_assert(kResWinVecs * 16 == 65536, "the buffer of a window is a bit above its 16-bit addresses");
static_assert((2 * kResWinVecs + 2 * kRecordRoom) * 16 <= 160 * 1024, "LDS of a CU");
static_assert(kResidueWindowRowsMax == 512 && kBlockItems == 32, "a plan entry holds 9 bits of window row and 5 of slot");

inline int window_grid(int m2) { return min(kWindowWgs, (plan_residue_chunks(m2) + kXcds - 1) / kXcds * kXcds); }

// The chunks of one workgroup: a contiguous share of the list per XCD, adjacent chunks to its
// workgroups at the same time (their windows overlap), chunks without a window left out.
struct ChunkWalk {
    int at, end, stride;
    __device__ __forceinline__ ChunkWalk(int m2)
    {
        const int chunks = plan_residue_chunks(m2), share = (chunks + kXcds - 1) / kXcds, xcd = blockIdx.x % kXcds;
        at = xcd * share + blockIdx.x / kXcds;
        end = min(chunks, (xcd + 1) * share);
        stride = gridDim.x / kXcds;
    }
    // the first one with a window from c on (end or later: none)
    __device__ __forceinline__ int from(const PlannedChunk* __restrict__ rows, int c) const
    {
        while (c < end && rows[c].wn <= 0) c += stride; // (the standard kernel has those)
        return c;
    }
};

__device__ __forceinline__ unsigned lds_address(const void* p)
{
    return (unsigned)(size_t)(const __attribute__((address_space(3))) char*)p;
}

// Copies 16 bytes per lane from base + offset to LDS at lds + 16 * lane, without a register in
// between.  The compiler does not know of the copy: copies_done waits for all of the wave's.
__device__ __forceinline__ void copy_to_lds(unsigned lds, const void* base, unsigned offset)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void copies_done()
{
    __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0)
}

// A chunk's record to LDS.
__device__ __forceinline__ void fetch_record(unsigned lds, const PlannedChunk* chunk, int wave)
{
    if (wave * kWave < kRecordVecs) copy_to_lds(lds + wave * kWave * 16, chunk, min((int)threadIdx.x, kRecordVecs - 1) * 16);
}

// One column tile of the window rows [0, wn) to LDS: `tile` points at it in the first row, rows are
// row_bytes apart (window_takes: 32-bit offsets), `at` is this lane's 16 bytes of a row (any valid place of it for a lane
// past the last column).
__device__ __forceinline__ void fetch_window(unsigned lds, const void* tile, unsigned row_bytes, int wn, unsigned at, int wave)
{
#pragma unroll
    for (int u = 0; u < kResidueWindowRowsMax / kPlanResidueChunk; ++u)
        if (u * kPlanResidueChunk + wave * (kWave / kResLanes) < wn) // (a wave's rows past the window: its last one again)
            copy_to_lds(lds + (u * kResThreads + wave * kWave) * 16, tile,
                        (unsigned)min(u * kPlanResidueChunk + (int)threadIdx.x / kResLanes, wn - 1) * row_bytes + at);
}

// One residue row as its lane group keeps it: cnt slots at positions 0 .. cnt - 1 (the order
// of the plan), the rest of the 32 positions carry value 0.
// addr[i]: the offsets in a window of this lane's 16 bytes of the dense rows of positions 2 i (low half)
// and 2 i + 1; for a position whose dense row is outside the window (its bit of missmask) it is that of
// one of the row's positions that is inside, and the data has to come from memory instead.
struct ResidueRow {
    int row;   // -1: nothing to do
    int first; // first residue slot of the row in column_indices / values
    int cnt;
    unsigned missmask;
    bool accumulate; // the row also has block segments (SpMM adds instead of storing)
    unsigned addr[kBlockItems / 2];
};

// The slot (counted from its row's first) that the plan put at position i of row `local` of a chunk.
__device__ __forceinline__ int planned_slot(const PlannedChunk& pc, int local, int i)
{
    return (pc.entry[local][i] >> 9) & (kBlockItems - 1);
}

// The lane group's view of its row (everything but the values).  skip_owned_slots: rows with block
// segments and at most that many aligned slots are left to the block kernel (SpMM under the whole-lists
// promise); 0 for SDDMM.
__device__ __forceinline__ void decode_planned_row(const PlannedChunk& pc, int local, int skip_owned_slots, ResidueRow& rr)
{
    const int ls = threadIdx.x % kResLanes;
    const int4 meta = *reinterpret_cast<const int4*>(&pc.meta[local]);
    const bool mine = meta.x >= 0 && !(((meta.z >> 8) & 1) && ((meta.z >> 16) & 0xffff) <= skip_owned_slots);
    rr.row = mine ? meta.x : -1;
    rr.first = mine ? meta.y : 0;
    rr.cnt = mine ? meta.z & 0xff : 0;
    rr.accumulate = (meta.z >> 8) & 1;
    rr.missmask = mine ? (unsigned)meta.w : 0u;
#pragma unroll
    for (int i = 0; i < kBlockItems / 8; ++i) {
        const uint4 e = reinterpret_cast<const uint4*>(pc.entry[local])[i];
        const unsigned w[4] = {e.x, e.y, e.z, e.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) // two entries at once
            rr.addr[4 * i + j] = ((w[j] & (0x10001u * (kResidueWindowRowsMax - 1))) * (kResLanes * 16)) | (0x10001u * 16 * ls);
    }
}

// Where position 2 i (odd = 0) or 2 i + 1 of a row is in the two windows: addr[i] unpacked, the buffer put above it.
template <int ODD>
__device__ __forceinline__ unsigned window_offset(unsigned pair, unsigned buffer_bit)
{
    return __builtin_amdgcn_perm(buffer_bit, pair, ODD ? 0x07060302u : 0x07060100u);
}

// ---- rings: the windows of a band's chunks one after the other -----------------------------------
// A workgroup that takes a contiguous strip of chunks finds most of a chunk's window in LDS already: the windows of neighbouring
// chunks overlap but for about as many rows as a chunk has.  Dense row r lies at row r % kRingRows of a ring; a chunk's new rows are
// copied during the one before, 1024 bytes a wave and copy.  TILES: 128-byte tiles that a row of the ring has (a dense row
// or a slice of one).  With two, those of odd rows change places: lane groups that read rows of different parity then meet in
// different banks here too.
//
// What bounds them: the window kernels copy every window whole, three times what a chunk of 128 rows is new in with a band of 256,
// and a copy has only the work on one tile to arrive in (500 K rows of 27, 32 doubles: 4.1 us a tile of which the LDS reads need 1.8).
// Here a chunk is one piece of work with one barrier, and its copies are a third and have all of it.  us, window kernels (standard
// kernels for rows of 128 bytes) -> rings, 27 slots a row and a band of 256: SpMM 500 K x 32 doubles 125 -> 108 (405 MB at 3.8 TB/s; a large
// copy would take 82), 1 M x 32 doubles 239 -> 200, 1 M x 64 233 -> 191, x 128 (two slices, by two workgroups side by side that share values and
// records in L2) 404 -> 346, x 128 halves 317 -> 274, 500 K x 16 doubles 125 -> 69, 1 M x 32 199 -> 141; SDDMM 1 M x 64 249 -> 222, x 128 halves 278
// -> 253, x 32 236 -> 171.  SDDMM of 512-byte rows keeps the window kernel: a row does not fit the ring, and its slices' sums meet.
constexpr int kRingRows = 512;
constexpr int kRingRecordVecs = (int)(sizeof(PlannedChunk) - offsetof(PlannedChunk, meta)) / 16; // (the window itself is read apart)
static_assert(offsetof(PlannedChunk, meta) == 16 && kRingRecordVecs % kWave == 0, "whole copies");
struct RingRecord {
    PlannedRowMeta meta[kPlanResidueChunk];
    unsigned short entry[kPlanResidueChunk][kBlockItems];
};
static_assert(sizeof(RingRecord) == kRingRecordVecs * 16, "the same");

__device__ __forceinline__ void fetch_ring_record(unsigned lds, const PlannedChunk* chunk, int wave)
{
    if (wave * kWave < kRingRecordVecs) copy_to_lds(lds + wave * kWave * 16, chunk->meta, threadIdx.x * 16u);
}

template <int TILES>
struct Ring {
    static constexpr int kRowBytes = 128 * TILES, kBytes = kRingRows * kRowBytes, kRowsPerCopy = 1024 / kRowBytes;
    // Dense rows [from, to) into the ring at `lds`; dense: this slice of row 0, row_bytes: of a whole row (at most 2^32 / 8).
    static __device__ __forceinline__ void fetch(unsigned lds, const char* dense, unsigned row_bytes, int from, int to, int wave, int lane)
    {
        const int r = lane * 16 / kRowBytes, tile = TILES == 1 ? 0 : (lane / 8 ^ r) & 1;
        const unsigned at = (unsigned)r * row_bytes + tile * 128u + lane % 8 * 16u;
        for (int first = (from / kRowsPerCopy + wave) * kRowsPerCopy; first < to; first += kResThreads / kWave * kRowsPerCopy)
            if (first + r >= from && first + r < to) // (a lane left out writes nothing)
                copy_to_lds(lds + (unsigned)(first % kRingRows) * kRowBytes, dense + (size_t)first * row_bytes, at);
    }
    // Where the first tile of this lane's 16 bytes of two window rows is, in units of 16 bytes (both halves of a pair of entries).
    static __device__ __forceinline__ unsigned units(unsigned entries, int w0, int ls)
    {
        const unsigned rows = ((entries & 0x01ff01ffu) + (unsigned)(w0 % kRingRows) * 0x10001u) & 0x01ff01ffu;
        return TILES == 1 ? rows * 8u + ls * 0x10001u : rows * 16u + ((rows & 0x10001u) << 3) + ls * 0x10001u;
    }
};

// A strip: chunks [at, end) one after the other, those without a window left out.  Of every XCD's share a strip per workgroup and slice, with as many
// chunks that have a window as the others: where some have none (`all` false) they are counted first, 64 descriptors a wave at a time.  (us, strips
// of as many chunks of any kind, each read on its own -> this, with the standard kernels for the others: 1 M rows of 27 x 64, half of the chunks
// with a window, those of an XCD's share together 659 -> 626, six in ten, eight runs a share 575 -> 549; eight in ten, 64 runs, 387 -> 398.)
struct RingWalk {
    int at, end, slice;
    // (room: kResThreads / kWave + 2 ints of LDS)
    __device__ __forceinline__ RingWalk(int m2, int slices, bool all, const int* __restrict__ plan, int* room)
    {
        const int chunks = plan_residue_chunks(m2), share = (chunks + kXcds - 1) / kXcds, xcd = blockIdx.x % kXcds;
        const int first = min(chunks, xcd * share), count = min(chunks, first + share) - first;
        const int strips = gridDim.x / kXcds / slices, strip = blockIdx.x / kXcds / slices;
        slice = blockIdx.x / kXcds % slices;
        if (all) {
            at = first + (int)((long long)count * strip / strips), end = first + (int)((long long)count * (strip + 1) / strips);
            return;
        }
        constexpr int kWaves = kResThreads / kWave;
        const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
        const int from = first + (int)((long long)count * wave / kWaves), to = first + (int)((long long)count * (wave + 1) / kWaves); // (this wave's)
        auto with_window = [&](int c) { return __ballot(c + lane < to && plan_residue_desc(plan, min(c + lane, chunks - 1)).wn > 0); };
        int mine = 0;
        for (int c = from; c < to; c += kWave) mine += __builtin_popcountll(with_window(c));
        if (lane == 0) room[wave] = mine;
        if (threadIdx.x < 2) room[kWaves + threadIdx.x] = first + count;
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            before += w < wave ? room[w] : 0;
            total += room[w];
        }
        const int bounds[2] = {(int)((long long)total * strip / strips), (int)((long long)total * (strip + 1) / strips)};
        for (int c = from; c < to; c += kWave) {
            const unsigned long long has = with_window(c);
            const int rank = before + __builtin_popcountll(has & ((1ull << lane) - 1ull));
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if ((has >> lane & 1) && rank == bounds[i]) room[kWaves + i] = c + lane;
            before += __builtin_popcountll(has);
        }
        __syncthreads();
        at = __builtin_amdgcn_readfirstlane(room[kWaves]), end = __builtin_amdgcn_readfirstlane(room[kWaves + 1]);
    }
    // the first chunk with a window from c on
    __device__ __forceinline__ int from(const PlannedChunk* __restrict__ rows, int c) const
    {
        while (c < end && rows[c].wn <= 0) c += max(rows[c].next, 1); // (the standard kernel has those)
        return min(c, end);
    }
};

// Longest row (in slot quads) among the 8 lane groups of the wave, as a scalar: quads at
// or past it are skipped by the whole wave.
__device__ __forceinline__ int wave_max_quads(int quads)
{
#pragma unroll
    for (int m = kResLanes; m < kWave; m <<= 1) quads = max(quads, __shfl_xor(quads, m, kWave));
    return __builtin_amdgcn_readfirstlane(quads);
}

} // namespace rode
