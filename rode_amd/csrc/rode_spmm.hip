// SpMM over a row-decomposed CSR matrix:  C[row, :] += sum_idx values[idx] * B[col(idx), :]
// Same work split, index arithmetic and store/accumulate rules as the
// reference's SparseKernel::Kernel4Block (RoDe_SpMM/RoDeSpmm.cu:197-476) and
// Kernel4Residue (:41-195); the execution shape is written for 64-lane
// wavefronts:
//
//   * the dense tile is TN columns wide; LPR = TN / (elements per 128-bit load)
//     lanes cover one B row, so one load instruction of a wave gathers 64 / LPR
//     different B rows, each as full 128-bit coalesced reads;
//   * (col, value) pairs of up to 64 nonzero slots are staged in LDS with one
//     coalesced load per lane and read back four at a time as broadcasts;
//   * block kernel: one wave per block segment; its lane groups take
//     interleaved slot quads, the partial rows are combined with a butterfly
//     over the groups and added to C with hardware fp32 atomics (always, as in
//     RoDeSpmm.cu:464-474: a long row has several segments and usually a residue).
//     Rows of 32..1024 slots are an exception in the execution, not in the result:
//     the wave of the row's first segment sums the whole row, tail included, and
//     adds it to C once; the row's other work items return at once;
//   * residue kernel: one group of LPR lanes per residue row, 64 / LPR rows per
//     wave (short rows are latency-bound and need many rows in flight); rows
//     shorter than 32 slots are stored with plain 128-bit stores, tails of
//     longer rows are added atomically (RoDeSpmm.cu:76-82, 173-194).
//
// Slots that belong to the previous row (the `start & 3` head of an unaligned
// segment) are neutralised with value 0 *and* the column of the first real slot,
// so a non-finite B row can never leak into a row that does not reference it
// (the reference multiplies B[0, :] by zero there, RoDeSpmm.cu:271-274).
#include "rode_items.hpp"
#include "rode_units.hpp"
#include "rode_internal.hpp"

#include <climits>
#include <type_traits>

namespace rode {

namespace {

// Rows of at most `owned_slots` aligned slots (and at least 32, i.e. rows that have block
// segments) are summed by a single wave of the block kernel (spmm_block_item).  The
// launcher passes kOwnedRowSlots when the caller promises that the two lists are the
// complete decomposition of the matrix (a row's first segment and its residue entry are
// then both in this call) and there are enough block segments to keep every CU busy
// anyway; else 0 (every work item on its own wave: small matrices need the parallelism
// more than they mind the extra atomics).  Measured on both sides: with 3936 segments
// (168 K nonzeros, width 128) the step takes 0.025 ms with whole rows and 0.030 ms without,
// with 9152 segments (1 M nonzeros, fp16 rows of 128) 0.104 against 0.120 ms; from 200 K
// segments on the difference is below 1 %.
constexpr int kOwnedRowSlots = 1024;
constexpr int kOwnedMinSegments = 1024;
// Where the caller knows that no row is longer than this, a matrix of fewer segments has its rows summed whole as well: a wave has no more
// than six steps to do, every row is stored, and C is not cleared beforehand (us, cleared and added to -> stored, widths 32 / 128 / 128 of
// halves: 512 x 512 of 16 to 64 nonzeros 8.2 - 9.8 -> 6.0 - 7.0, 8000 of 24 x 128 14.7 -> 10.3, of halves 13.2 -> 6.5, 40 K of 16 x 64 17.3
// -> 15.0, 250 K 150 -> 143; longest row 168 7.7 / 10.6 / 12.0 -> 5.7 / 6.0 / 5.7, 227 7.8 / 9.8 / 10.7 -> 5.7 / 6.4 / 5.7, 338 7.5 / 8.7 /
// 9.0 -> 5.8 / 7.3 / 6.7, 471 7.9 / 9.9 / 10.4 -> 5.8 / 9.1 / 7.8, 502 8.4 / 8.4 / 8.2 -> 5.9 / 9.4 / 8.2, 1001 7.4 / 8.5 / 7.9 -> 8.0 /
// 15.0 / 12.6). Each 64 slots of such a row have a sum of their own, as the row's segments had: one chain over all of a row had up to 1.7
// times their error.
constexpr int kShortRowSlots = 384;
// Without the promise the block kernel may still merge the short segments of a row that
// the list it was given holds, when there are this many of them.
constexpr int kMergeMinSegments = 16384;
// Rows longer than one wave sums (kOwnedRowSlots), where C is not cleared: the four waves of a workgroup sum such a row, a quarter each with the
// tail in it, the sums meet in LDS and the row is stored.  Adding to it, segment by segment, takes C cleared before, a launch of 3 to
// 5 us that reads every row offset.  The workgroup is the first whose four segments are all the row's (there is one among any seven
// consecutive ones); a row that has none is summed by the wave of its first segment, whatever its length.
// Where it pays (us, cleared and added to -> stored; lognormal degrees, rows of mean degree x width, longest row L): what a row of L slots
// takes - 1.1 to 1.6 ns a slot on an idle GPU with tiles of 128 bytes, 2 with 256, 4.5 with 512, 3.5 in a large matrix - is nowhere to be seen
// while the others take longer.
//   * L up to 4096: 16 K of 16 x 64 17.1 -> 13.8 (L 2603), 25 K of 10 x 32 11.8 -> 8.3, 36 K of 10 halves x 32 12.5 -> 8.9, 30 K of 24 halves x 128
//     24.7 -> 20.9, 42 K of 15 x 128 34.7 -> 31.3, 65 K of 16 x 128 60.3 -> 57.0, 100 K of 16 x 64 52.8 -> 49.6 (3349); above it, with less than
//     300 MB of dense rows to gather: 36 K of 22 halves x 64 18.8 -> 24.8 (6973), 20 K of 26 x 96 25.0 -> 26.4 (5736), 16 K of 32 halves x 32
//     13.1 -> 11.9 (5206).  Up to 3072 for tiles of 256 bytes (8000 rows of 40 halves x 128, L 2000 14.7 -> 12.1, 3000 14.8 -> 14.6, 4000 15.2 -> 16.8;
//     3000 x 64 2000 11.0 -> 7.3, 3000 11.5 -> 9.4, 4000 11.5 -> 11.1), 2048 of 512 (8000 x 128 2000 20.3 -> 19.4, 3000 20.9 -> 24.9);
//   * L up to 6656 from 300 MB on: 27 K of 26 x 128 33.4 -> 29.4 (5640), 59 K of 30 halves x 128 52.8 -> 47.8 (6141), 51 K of 19 x 128 50.1 -> 47.6
//     (6677); 29 K of 32 x 128 40.4 -> 41.9 (7741).  Above 666 MB a slot for every 100 KB, up to the 20 000 that have been measured: 100 K of 24 x 128
//     (1.2 GB) 152.2 -> 146.8 (12 000), 300 K of 16 (2.4 GB) 363.6 -> 363.4 (12 000), 383.3 -> 382.5 (20 000), 400 K (3.3 GB) 493 -> 491 (20 000), of 24
//     (4.8 GB) 682 -> 688 (12 000), 686 -> 691 (20 000), of halves 368.5 either way;
//   * segments of more than 128 slots, whose rows of up to six segments may have no workgroup, from 500 MB on: 200 K of 16 x 64 120.4 -> 116.5,
//     150 K x 128 167 -> 163, 180 K of 20 halves x 128 135 -> 132; 113 K of 23 x 32, 332 MB, 44.7 -> 49.6.
// 2-norms of the long rows' errors against fp64, relative to adding their segments up (which were merged to 512 slots as well): 0.97 to 1.006,
// rows of 1100 to 6500, widths 32 to 128, both types.
// Not above 6656 slots with partial tiles, whose matrices have B past the L2s and no tiles of one line (30 K of 110 x 100 154 -> 166, x 112 165 -> 177, 60 K
// of 60 x 100 212 -> 224, of 110 x 56 202 -> 213).
inline bool wide_rows_pay(int longest, int seg_length, size_t tile_bytes, size_t gathered, bool partial)
{
    constexpr size_t MB = 1000000;
    if (seg_length > (gathered >= 500 * MB ? 512 : 128)) return false;
    if (gathered < (tile_bytes > 256 ? 500 : 300) * MB) return longest <= (tile_bytes > 256 ? 2048 : tile_bytes > 128 ? 3072 : 4096);
    return (size_t)longest <= (partial ? (size_t)6656 : min(max((size_t)6656, gathered / 100000), (size_t)20000));
}

// Up to this many workgroups, and when both kernels go to the same stream, the two lists
// are processed by one launch (spmm_pair_kernel).  Above it the residue kernel runs on its
// own: it needs a quarter of the block kernel's registers and keeps twice the waves per CU.
// (Sharded launches, below, keep to one launch for longer: their workgroups are smaller.  Power-law-like
// rows, 65 K x 65 K, 1 M nonzeros, width 128: 75 us in two launches, 63 in one.)
constexpr int kPairMaxWorkgroups = 16384;
constexpr int kPairMaxSharded = 65536;
// Residue rows alone, with the rows without slots of an uncleared C: up to this many (a clearing launch costs 2 to 3 us: 512 rows of 4 x 64
// 8.4 -> 6.3, 16 K of 8 x 128 9.9 -> 7.8, 100 K of 8 x 32 18.6 -> 16.4, 40 K of 8 halves x 128 14.7 -> 12.5), then the residue kernel, which
// has more waves per CU, with a launch before it.
constexpr int kPairMaxAlone = 4096;

// Sharding.  Every XCD has an L2 of its own (4 MB), and rows of B that are referenced at random are
// fetched into all eight.  When a row of B is 2, 4 or 8 lines of 128 bytes, C is computed in column
// tiles of one line and XCD x works on tile x mod lines only: of B it sees one line per row, so that a
// matrix of up to lines x 4 MB stays in the L2s, and of twice that about half of it does.  The nonzeros'
// columns and values are read once per tile (8 bytes against 128 gathered), and every work item is there once per tile.
// Rows whose columns lie close together share their lines without it (band of 256 in 60 K rows: 32 -> 39).
//
// Where it pays (us unsharded -> sharded; dense rows x width, nonzeros per row drawn from a Poisson (p) or a lognormal (l) distribution):
//   * B above 4 MB, which one L2 does not hold: l 16 K x 128 of 16: 26.7 -> 17.3, 65 K x 128 72 -> 59, 65 K x 64 36.8 -> 32.6; 8.5 K x 128
//     (4.4 MB) p of 8 5.5 -> 5.9, of 16 10.7 -> 10.0;
//   * up to 26 MB per tile, where half of a tile and more misses the L2 (l of 16: 200 K x 64 126 -> 120, x 128 243 -> 235; p 212 K x 64
//     124 -> 128, 400 K x 64 472 -> 492), up to 14 MB with eight tiles (l of 16: 100 K x 256 228 -> 211, 150 K 339 -> 347, 200 K 463 -> 490);
//   * where a row of B is used less than six times: from 12 MB up to 9 MB per tile (p of 4: 33 K x 64 8.4 -> 8.9, 33 K x 128 15.2 -> 13.1,
//     65 K x 128 26.6 -> 23.9, 150 K 54.1 -> 56.2; p of 2: 65 K 19.1 either way, 150 K 37.4 -> 40.2);
//   * where many rows have a block segment beside their tail (p of 28 and more): twice the work items, and more of B has to miss.
//     Work items of 24 nonzeros and more: from 8 MB on, 16 with eight tiles, 48 with halves (p of 64: 12 K x 128 26.5 -> 29.0,
//     16 K x 128 43.4 -> 38.5, 24 K x 64 28.1 -> 28.9, 33 K x 64 45.1 -> 39.0, 8.5 K x 256 34.0 -> 38.7, 16 K x 256 84 -> 75, 16 K x 512 halves
//     69 -> 82, of 50 33 K 155 -> 167, 65 K 382 -> 354).  Smaller ones: from 16 MB on, 32 with eight tiles (p of 40: 12 K x 128 23.6 -> 30.0,
//     24 K 54.8 -> 56.4, 33 K 79.3 -> 76.3, 33 K x 64 37.0 -> 40.3, 65 K x 64 83 -> 76, 24 K x 256 104 -> 108, 65 K x 256 336 -> 297), not with
//     halves (p of 36, x 128: 65 K 79.8 -> 82.7, 150 K 188 -> 199; of 40, x 512: 65 K 316 -> 336).
// items: of both lists; segments: do many rows have one; nonzeros: 0 when the caller did not say.
inline bool sharding_pays(int lines, bool halves, size_t dense_rows, long long items, bool segments, long long nonzeros)
{
    constexpr size_t MB = (size_t)1 << 20;
    const size_t tile = dense_rows * 128, bytes = tile * lines;
    if (tile > (lines == 8 ? 14 : 26) * MB || bytes <= 4 * MB) return false;
    if (nonzeros > 0 && (size_t)nonzeros < 6 * dense_rows && (tile > 9 * MB || bytes < 12 * MB)) return false;
    if (!segments) return true;
    if (nonzeros > 0 && nonzeros < 24 * items) return !halves && bytes >= (lines == 8 ? 32 : 16) * MB;
    return bytes >= (lines < 8 ? 8 : halves ? 48 : 16) * MB;
}

// Sum over the aligned slots [base, base + cnt) of values * B rows, for this lane's columns
// of the tile; the first `mask` slots (the previous row's) and the slots past cnt in the
// last quad are neutralised.  Every lane of the wave returns the wave's total.
// (split, jump: the slots are [base, base + split) followed by [base + split + jump, ...):
// a row with a hole that somebody else works on; split >= cnt for one plain range.)
// PART: so many slots (0: all) have a sum of their own, and the total is the sum of those (more than one step's: kept in LDS, in this
// lane's place `parked`; in registers they cost the kernel of 32-column tiles a wave per SIMD).  EIGHTS: see spmm_gather.
template <typename T, int TN, int PART = 0, bool EIGHTS = false>
__device__ __forceinline__ void spmm_sum_slots(int base, int mask, int cnt, int split, int jump, int lane, int* my_c,
                                               typename DenseVec<T>::Acc* my_v, const T* b_lane, int n,
                                               const int* __restrict__ col,
                                               const typename DenseVec<T>::Acc* __restrict__ val,
                                               typename DenseVec<T>::Acc (&total)[SpmmShape<T, TN>::kVec],
                                               typename DenseVec<T>::Acc* parked = nullptr)
{
    using S = SpmmShape<T, TN>;
    using A = typename S::Acc;
    constexpr int VEC = S::kVec, LPR = S::kLpr, G = S::kGroupsWave;
    const int group = lane / LPR;
    A acc[VEC], parts[VEC];
#pragma unroll
    for (int x = 0; x < VEC; ++x) acc[x] = parts[x] = A(0);

    // slots of the previous row (head) and slots past the end (last quad) are neutralised:
    // value 0, column of a real slot
    auto fetch = [&](int off, int& c, A& v) __attribute__((always_inline)) {
        const int slot = off + lane;
        if (lane < ((min(cnt - off, kWave) + 3) & ~3)) {
            const int at = min(max(slot, mask), cnt - 1);
            const int idx = base + at + (at >= split ? jump : 0);
            c = col[idx];
            v = val[idx];
        }
    };
    int c = 0;
    A v = A(0);
    fetch(0, c, v);
    static_assert(PART % kWave == 0, "whole steps");
    for (int off = 0, end = PART > kWave ? min(PART, cnt) : cnt;;) {
    for (; off < end; off += kWave) {
        const int slot = off + lane;
        const int live = min(cnt - off, kWave); // 64, or less on the last step
        my_c[lane] = c;
        my_v[lane] = slot < mask || slot >= cnt ? A(0) : v;
        wave_lds_sync();
        // (on its way while the dense rows arrive: power law 2 M x 128 3620 -> 3600 us, 1 M x 32 545 -> 520, 300 K x 128 626 -> 609, of
        // halves 368 -> 351; lognormal 20 K x 64 19.8 -> 16.9, 65 K x 128 either way; 16 K rows of 100, width 64 25.8 -> 24.6)
        if (off + kWave < cnt) fetch(off + kWave, c, v);
        if (live == kWave)
            spmm_gather<T, TN, 16 / G, true, EIGHTS>(b_lane, (size_t)n, acc, my_c, my_v, group, G, 16);
        else
            spmm_gather<T, TN, 16 / G, false, EIGHTS>(b_lane, (size_t)n, acc, my_c, my_v, group, G, (live + 3) / 4);
        if constexpr (PART == kWave) {
#pragma unroll
            for (int x = 0; x < VEC; ++x) parts[x] += acc[x], acc[x] = A(0);
        }
        wave_lds_sync();
    }
    if (PART <= kWave || off >= cnt) break;
#pragma unroll
    for (int x = 0; x < VEC; ++x) parked[x] = off > PART ? parked[x] + acc[x] : acc[x], acc[x] = A(0);
    end = min(off + PART, cnt);
    }
#pragma unroll
    for (int x = 0; x < VEC; ++x) {
        if (PART > kWave && cnt > PART) acc[x] += parked[x];
        total[x] = butterfly_sum<LPR, kWave>(PART == kWave ? parts[x] : acc[x]);
    }
}

// Calls of widths that are a multiple of 32 and not of 128 may take tiles of 128 or 64 columns for tiles of 32 (spmm_tile_of_call), with 2 or 4 times
// fewer lane groups for a row's slots: their sums are made of sums of eight slots.  2-norms of the errors against fp64 relative to tiles of 32
// (uniform, width 96): one chain a lane group, 40 nonzeros a row 1.31, halves 1.09, 110 halves 1.38; like this, 34 to 110 nonzeros 0.97 to 1.004,
// halves 0.985 to 1.001.  Time (us, chain -> this): 4000 rows of 56 7.1 -> 7.2, 60 K of 56 119 -> 119, halves
// 8000 of 110 11.9 -> 12.2, 16.5 K of 56 17.0 -> 17.2.
// (Not for other widths, which had tiles of that many columns before: lognormal 100 K of 30 x 48 93 -> 100 us, 12 K of 14 14.3 -> 15.7.)
constexpr int kPartialEights = 2; // (EDGE: the last tile is partial (kPartial), and so the sums are)
template <int EDGE>
constexpr bool kInEights = EDGE == kPartialEights;

// Which column tile of C, and which of the `blocks` workgroups of its grid row, a workgroup is.
// shards == 1: tiles in blockIdx.y.  shards > 1 (a divisor of kXcds): XCD x only ever works on tile
// x % shards, its grid rows dealt out one after the other in a one-dimensional grid.
struct TilePlace {
    int bid, tile;
};
__device__ __forceinline__ TilePlace tile_place(int b, int blocks, int shards)
{
    if (shards == 1) return TilePlace{b, (int)blockIdx.y};
    const int x = b % kXcds, at = x / shards * (blocks / kXcds * shards) + b / kXcds; // position in the tile's row, contiguous per XCD
    // (as the id that xcd_logical_block takes to that position)
    return TilePlace{at % (blocks / kXcds) * kXcds + at / (blocks / kXcds), x % shards};
}

// The work item of the wave of segment `seg` (of a workgroup that has kWavesPerWg consecutive ones) where workgroups take long rows
// (wide_rows_pay); not whole: a quarter of the row.
__device__ __forceinline__ bool spmm_wide_item(int seg, int m1, int owned_slots, const int* __restrict__ block_rows, const int* __restrict__ row_ptr,
                                               BlockItem& it)
{
    const int row = block_rows[seg];
    const int row_start = row_ptr[row], row_end = row_ptr[row + 1], mask = row_start & (kVecLen - 1), base = row_start - mask;
    const bool first = seg == 0 || block_rows[seg - 1] != row;
    it.row = row, it.mask = mask, it.base = base, it.cnt = row_end - base, it.whole = true;
    if (it.cnt <= owned_slots) return first;
    auto all_of = [&](int s) { return s >= 0 && s + kWavesPerWg <= m1 && block_rows[s] == row && block_rows[s + kWavesPerWg - 1] == row; };
    const int mine = seg / kWavesPerWg * kWavesPerWg;
    if (all_of(mine)) {
        if (mine > 0 && all_of(mine - kWavesPerWg)) return false; // (the workgroup before has the row)
        const int each = (it.cnt + kWavesPerWg * kWave - 1) / (kWavesPerWg * kWave) * kWave, from = (seg - mine) * each;
        it.base = base + from, it.mask = from == 0 ? mask : 0, it.cnt = min(each, it.cnt - from), it.whole = false;
        return true;
    }
    return first && !all_of(seg == mine ? mine : mine + kWavesPerWg);
}

// One wave per block segment (see sddmm_block_kernel for the slot arithmetic,
// identical at RoDeSpmm.cu:210-234).
// (bid of nblocks: the workgroup's position in the part of the grid that works on block segments)
// WALK: 0 one wave per segment only, 1 chunks only (chunk_hint > 1), 2 either, found out here; 3 one wave per segment, which
// sums its row in parts (kShortRowSlots); 4 (with STORE) one per segment too, and a workgroup for a row of more than owned_slots (wide_rows_pay).
// (Kernels of their own, so that the code of one way does not cost the other registers.)
// STORE: a row's only work item stores its sum instead of adding it (owners.overwrite; a
// kernel of its own as well: as a run-time branch it slowed the fp16 kernel of width 128
// that never takes it from 0.97 to 1.13 ms on the power-law benchmark).
template <typename T, int TN, int EDGE, int WALK, bool STORE>
__device__ __forceinline__ void
spmm_block_body(int bid, int nblocks, int tile, int m1, int n, int owned_slots, int chunk_hint, RowOwners owners,
                const int* __restrict__ block_rows,
                const int* __restrict__ st_off, const int* __restrict__ row_ptr, const int* __restrict__ col,
                const typename DenseVec<T>::Acc* __restrict__ val, const T* __restrict__ B,
                typename DenseVec<T>::Acc* __restrict__ C)
{
    using S = SpmmShape<T, TN>;
    using A = typename S::Acc;
    constexpr int VEC = S::kVec, LPR = S::kLpr, G = S::kGroupsWave;
    __shared__ __attribute__((aligned(16))) int lds_c[kWavesPerWg * kWave];
    __shared__ __attribute__((aligned(16))) A lds_v[kWavesPerWg * kWave];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave; // (uniform: scalar registers)
    // Lists with short segments (and enough of them that merging is on): a wave walks a chunk
    // of consecutive segments from leader to leader, adds up what it finds for one row and
    // updates that row of C once (the sums of the items, not one long sum: same rounding as
    // the combine of neighbouring waves below).
    int chunk = 1;
    if constexpr (WALK == 1) chunk = chunk_hint;
    if constexpr (WALK == 2)
        chunk = block_chunk_for_grid(owned_slots != 0 && m1 >= kWalkMinSegments ? block_chunk(m1, block_rows, st_off) : 1, m1,
                                     nblocks);
    if (WALK != 0 && WALK < 3 && chunk > 1) {
        const long long first = chunk_first_segment(bid, wave, m1, chunk);
        if (first < 0) return;
        const int last = (int)min(first + chunk, (long long)m1);
        const int ls = lane % LPR, group = lane / LPR;
        const bool col_ok = !EDGE || tile + ls * VEC < n;
        const T* b_lane = B + tile + (col_ok ? ls * VEC : 0);
        constexpr int EPG = VEC / G > 0 ? VEC / G : 1; // elements each lane group adds to C
        A row_total[VEC];
        int pending = -1;           // the row that row_total belongs to
        bool pending_whole = false; // ... is that row's one work item
        auto flush = [&]() {
            A* c_lane = C + (size_t)pending * n + tile + ls * VEC;
            if (STORE && pending_whole) { // (the same in every lane)
#pragma unroll
                for (int x = 0; x < VEC; ++x)
                    if (group == x / EPG && col_ok) c_lane[x] = row_total[x];
                return;
            }
#pragma unroll
            for (int x = 0; x < VEC; ++x)
                if (group == x / EPG && col_ok) atomicAdd(c_lane + x, row_total[x]);
        };
        for (int from = (int)first; from < last; from += kScanSegments) {
            const ChunkScan scan = scan_chunk(kSpmmMergeSlots, from, m1, owned_slots, owners, lane, block_rows, st_off, row_ptr);
            const int count = min(last - from, kScanSegments);
            for (unsigned long long todo = scan.items & ((1ull << count) - 1ull); todo; todo &= todo - 1ull) {
                const BlockItem it = chunk_item(scan, __builtin_ctzll(todo));
                A total[VEC];
                spmm_sum_slots<T, TN, 0, kInEights<EDGE>>(it.base, it.mask, it.cnt, it.cnt, 0, lane, lds_c + wave * kWave, lds_v + wave * kWave,
                                      b_lane, n, col, val, total);
                if (it.row != pending) {
                    if (pending >= 0) flush();
                    pending = it.row;
                    pending_whole = it.whole;
#pragma unroll
                    for (int x = 0; x < VEC; ++x) row_total[x] = total[x];
                } else {
#pragma unroll
                    for (int x = 0; x < VEC; ++x) row_total[x] += total[x];
                }
            }
        }
        if (pending >= 0) flush();
        return;
    }
    const int seg0 = xcd_logical_block(bid, nblocks) * kWavesPerWg;
    const int seg = seg0 + wave;
    BlockItem it{-1, 0, 0, 0};
    const bool active = seg < m1 && (WALK == 4 ? spmm_wide_item(seg, m1, owned_slots, block_rows, row_ptr, it)
                                               : spmm_block_item(seg, m1, owned_slots, owners, lane, block_rows, st_off, row_ptr, it));
    // A wave without a work item leaves at once (with the reference's 32-slot segments that
    // is most waves); the barrier below then counts only the waves that are still running
    // (S_BARRIER waits on the surviving waves of a workgroup).
    if (!active) return;
    // Do two work items of this workgroup add to the same row (neighbouring segments of a
    // long row that are not merged into one leader)?  Every wave finds the same answer.  If
    // so, the waves add their sums up in LDS and the row of C gets one update per run of
    // such work items instead of one each.
    int item_row[kWavesPerWg]; // the row of each wave's work item, -1: that wave has none (and has left)
    bool shared_row = false;
    if constexpr (WALK == 4) {
        shared_row = !it.whole;
#pragma unroll
        for (int i = 0; i < kWavesPerWg; ++i) item_row[i] = it.row; // (of a row that is shared)
    }
#pragma unroll
    for (int i = 0; WALK != 4 && i < kWavesPerWg; ++i) {
        item_row[i] = spmm_block_leader_row(seg0 + i, m1, owned_slots, owners, block_rows, st_off, row_ptr);
        if (i > 0) shared_row = shared_row || (item_row[i] >= 0 && item_row[i] == item_row[i - 1]);
    }
    const int row = it.row, mask = it.mask, base = it.base, cnt = it.cnt;

    const int ls = lane % LPR, group = lane / LPR;
    // EDGE: n is not a multiple of TN; lanes past the last column re-read the tile's
    // first columns (a valid address) and never write
    const bool col_ok = !EDGE || tile + ls * VEC < n;
    const T* b_lane = B + tile + (col_ok ? ls * VEC : 0);
    int* my_c = lds_c + wave * kWave;
    A* my_v = lds_v + wave * kWave;

    // combine the lane groups, then spread the atomics over them
    constexpr int EPG = VEC / G > 0 ? VEC / G : 1; // elements each group adds
    constexpr int kPart = WALK == 3 ? kWave : WALK == 4 ? kSpmmMergeSlots : 0;
    A total[VEC];
    __shared__ __attribute__((aligned(16))) A parked[kPart > kWave ? kWgThreads * VEC : 1];
    spmm_sum_slots<T, TN, kPart, kInEights<EDGE>>(base, mask, cnt, cnt, 0, lane, my_c, my_v, b_lane, n, col, val, total, parked + (kPart > kWave ? threadIdx.x * VEC : 0));
    if (shared_row) {
        __shared__ __attribute__((aligned(16))) A wg_sum[kWavesPerWg][TN];
        if (group == 0) {
#pragma unroll
            for (int x = 0; x < VEC; ++x) wg_sum[wave][ls * VEC + x] = total[x];
        }
        __syncthreads();
        // the first wave of a run of equal rows takes the sums of the others
        bool first_of_run = true, run_goes_on = true;
#pragma unroll
        for (int w = 0; w < kWavesPerWg; ++w) {
            if (w + 1 == wave && item_row[w] == row) first_of_run = false;
            if (w > wave) {
                run_goes_on = run_goes_on && item_row[w] == row;
                if (run_goes_on && first_of_run) {
#pragma unroll
                    for (int x = 0; x < VEC; ++x) total[x] += wg_sum[w][ls * VEC + x];
                }
            }
        }
        if (!first_of_run) return;
    }
    A* c_lane = C + (size_t)row * n + tile + ls * VEC;
    if (STORE && (WALK == 4 || it.whole)) { // the row's only work item (the same in every lane): nothing to add to
#pragma unroll
        for (int x = 0; x < VEC; ++x)
            if (group == x / EPG && col_ok) c_lane[x] = total[x];
        return;
    }
#pragma unroll
    for (int x = 0; x < VEC; ++x)
        if (group == x / EPG && col_ok) atomicAdd(c_lane + x, total[x]);
}

// One group of LPR lanes per residue row (tail selection: RoDeSpmm.cu:71-82); the
// group walks its row's slot quads one after the other, no cross-lane reduction.
template <typename T, int TN, int EDGE>
__device__ __forceinline__ void
spmm_residue_body(int bid, int nblocks, int tile, int m2, int n, int owned_slots, RowOwners owners,
                  const int* __restrict__ residue_rows,
                  const int* __restrict__ row_ptr, const int* __restrict__ col,
                  const typename DenseVec<T>::Acc* __restrict__ val, const T* __restrict__ B,
                  typename DenseVec<T>::Acc* __restrict__ C, const int* __restrict__ plan)
{
    using S = SpmmShape<T, TN>;
    using A = typename S::Acc;
    constexpr int VEC = S::kVec, LPR = S::kLpr;
    constexpr int RPW = kWave / LPR;        // rows per wave
    constexpr int OWN = kBlockItems / LPR;  // slots staged by one lane
    // (16 bytes between the rows of a wave: its groups read their slots at the same time, from banks of their own)
    constexpr int kStrideC = kBlockItems + 4, kStrideV = kBlockItems + 16 / (int)sizeof(A);
    __shared__ __attribute__((aligned(16))) int lds_c[kWavesPerWg * RPW * kStrideC];
    __shared__ __attribute__((aligned(16))) A lds_v[kWavesPerWg * RPW * kStrideV];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave; // (uniform: scalar registers)
    const int group = lane / LPR, ls = lane % LPR;
    const int item = (xcd_logical_block(bid, nblocks) * kWavesPerWg + wave) * RPW + group;
    if (item >= m2) return;

    if (plan && plan_residue_desc(plan, item / kPlanResidueChunk).wn > 0) return; // the window kernel has this chunk

    const int row = residue_rows[item];
    const ResidueItem it = residue_item(row, row_ptr);
    const bool accumulate = it.accumulate; // the row also has block segments
    if (accumulate && it.aligned <= owned_slots) return; // summed entirely, tail included, by the block kernel
    if (owned_elsewhere(owners, row, it.aligned)) return; // another kernel has the whole row
    const int first = it.first, cnt = it.cnt;

    const bool col_ok = !EDGE || tile + ls * VEC < n;
    int* my_c = lds_c + (wave * RPW + group) * kStrideC;
    A* my_v = lds_v + (wave * RPW + group) * kStrideV;

    A acc[VEC];
#pragma unroll
    for (int x = 0; x < VEC; ++x) acc[x] = A(0);

    if (cnt > 0) {
        const int padded = (cnt + 3) & ~3; // slots past the tail repeat its last column with value 0
        int c[OWN];
        A v[OWN]; // (all of them on their way before the first is waited for)
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
            const int slot = ls + i * LPR, at = first + min(slot, cnt - 1);
            if (slot < padded) {
                c[i] = col[at];
                v[i] = val[at];
            }
        }
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
            const int slot = ls + i * LPR;
            if (slot < padded) {
                my_c[slot] = c[i];
                my_v[slot] = slot < cnt ? v[i] : A(0);
            }
        }
        wave_lds_sync();
        // (two quads in flight where their dense rows fit 32 registers: config 4 K=64 0.550 -> 0.535 ms, K=32
        // 0.305 -> 0.292; with fp16's eight elements per load it costs waves per SIMD instead: 0.66 -> 0.76 ms)
        if constexpr (VEC <= 4)
            spmm_gather_pairs<T, TN, kBlockItems / 4>(B + tile + (col_ok ? ls * VEC : 0), (size_t)n, acc, my_c, my_v, padded / 4);
        else
            spmm_gather<T, TN, kBlockItems / 4, false>(B + tile + (col_ok ? ls * VEC : 0), (size_t)n, acc, my_c, my_v, 0, 1,
                                                       padded / 4);
    }

    A* c_lane = C + (size_t)row * n + tile + ls * VEC;
    if (!col_ok) return;
    if (accumulate) {
#pragma unroll
        for (int x = 0; x < VEC; ++x) atomicAdd(c_lane + x, acc[x]);
    } else {
        store_row<VEC>(c_lane, acc);
    }
}

template <typename T, int TN, int EDGE, int WALK, bool STORE>
__global__ void __launch_bounds__(kWgThreads)
spmm_block_kernel(int shards, int m1, int n, int owned_slots, int chunk_hint, RowOwners owners, const int* __restrict__ block_rows,
                  const int* __restrict__ st_off,
                  const int* __restrict__ row_ptr, const int* __restrict__ col,
                  const typename DenseVec<T>::Acc* __restrict__ val, const T* __restrict__ B,
                  typename DenseVec<T>::Acc* __restrict__ C)
{
    const TilePlace at = tile_place(blockIdx.x, gridDim.x / shards, shards);
    spmm_block_body<T, TN, EDGE, WALK, STORE>(at.bid, gridDim.x / shards, at.tile * TN, m1, n, owned_slots, chunk_hint, owners, block_rows, st_off,
                                       row_ptr, col, val, B, C);
}

template <typename T, int TN, int EDGE>
__global__ void __launch_bounds__(kWgThreads)
spmm_residue_kernel(int shards, int m2, int n, int owned_slots, RowOwners owners, const int* __restrict__ residue_rows,
                    const int* __restrict__ row_ptr, const int* __restrict__ col,
                    const typename DenseVec<T>::Acc* __restrict__ val, const T* __restrict__ B,
                    typename DenseVec<T>::Acc* __restrict__ C, const int* __restrict__ plan)
{
    const TilePlace at = tile_place(blockIdx.x, gridDim.x / shards, shards);
    spmm_residue_body<T, TN, EDGE>(at.bid, gridDim.x / shards, at.tile * TN, m2, n, owned_slots, owners, residue_rows, row_ptr, col, val, B,
                                   C, plan);
}

// The rows of C without slots, which are in neither list, where nobody cleared C: 64 at a time to the waves, whose lanes zero the tile of
// several rows at once, 16 bytes each.  (A matrix may be mostly such rows: in waves of 256 that took one after the other, 100 K x 128 with
// 50 rows that are not empty took 29.4 us instead of 12.8 with a clearing launch, 1 M x 32 34 instead of 22.)
template <typename A, int TN, int EDGE>
__device__ __forceinline__ void spmm_empty_rows(int bid, int nblocks, int tile, int rows, int n, const int* __restrict__ row_ptr, A* __restrict__ C)
{
    constexpr int VEC = 16 / (int)sizeof(A), LPR = TN / VEC, AT_ONCE = kWave / LPR;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int group = lane / LPR, at = tile + lane % LPR * VEC;
    for (long long from = ((long long)bid * kWavesPerWg + wave) * kWave; from < rows; from += (long long)nblocks * kWgThreads) {
        const int mine = (int)min(from + lane, (long long)rows - 1);
        const int start = row_ptr[mine];
        const unsigned long long empty = __ballot(from + lane < rows && row_ptr[mine + 1] - start + (start & (kVecLen - 1)) <= 0);
        if (empty == 0) continue;
        A* to = C + (size_t)(from + group) * n + at;
#pragma unroll 4
        for (int i = 0; i < kWave; i += AT_ONCE, to += (size_t)AT_ONCE * n)
            if ((empty >> (i + group) & 1) && (!EDGE || at < n)) *reinterpret_cast<uint4*>(to) = make_uint4(0, 0, 0, 0);
    }
}
inline int empty_row_workgroups(int rows) { return (min((rows + kWgThreads - 1) / kWgThreads, 16384) + kXcds - 1) / kXcds * kXcds; }

// Both lists in one launch: the first g1 workgroups of a grid row (of every tile of a sharded
// grid) work on block segments, the others on residue rows.  For matrices so small that a launch costs as much as its
// kernel (a kernel of a few microseconds); the two parts then also fill the GPU together.
// g0 > 0 (with STORE: every other row is stored): as many workgroups after them zero the rows without slots.
template <typename T, int TN, int EDGE, int WALK, bool STORE>
__global__ void __launch_bounds__(kWgThreads)
spmm_pair_kernel(int shards, int g0, int rows, int g1, int m1, int m2, int n, int owned_slots, int chunk_hint, RowOwners owners,
                 const int* __restrict__ block_rows,
                 const int* __restrict__ residue_rows, const int* __restrict__ st_off, const int* __restrict__ row_ptr,
                 const int* __restrict__ col, const typename DenseVec<T>::Acc* __restrict__ val,
                 const T* __restrict__ B, typename DenseVec<T>::Acc* __restrict__ C, const int* __restrict__ plan)
{
    const int lists = gridDim.x - (STORE ? g0 * shards : 0);
    if (STORE && (int)blockIdx.x >= lists) {
        const TilePlace at = tile_place(blockIdx.x - lists, g0, shards);
        spmm_empty_rows<typename DenseVec<T>::Acc, TN, EDGE>(at.bid, g0, at.tile * TN, rows, n, row_ptr, C);
        return;
    }
    const bool segments = (int)blockIdx.x < g1 * shards;
    const int g = segments ? g1 : lists / shards - g1;
    const TilePlace at = tile_place(segments ? blockIdx.x : blockIdx.x - g1 * shards, g, shards);
    if (segments)
        spmm_block_body<T, TN, EDGE, WALK, STORE>(at.bid, g, at.tile * TN, m1, n, owned_slots, chunk_hint, owners, block_rows, st_off, row_ptr, col, val,
                                        B, C);
    else
        spmm_residue_body<T, TN, EDGE>(at.bid, g, at.tile * TN, m2, n, WALK == 4 ? INT_MAX : max(owned_slots, 0), owners, residue_rows,
                                       row_ptr, col, val,
                                       B, C, plan);
}

// The groups of a group plan (rode_group.hip): four adjacent rows with runs of consecutive
// columns that overlap in a long shared run (shared_run).  One wave per group (WPG = 1), or a
// workgroup whose four waves split the shared run.  Every dense row of it is loaded once
// and multiplied into the sums of all four rows (its address follows from the run, no
// column index is read).  Then the rows' other nonzeros: with one wave per group, of the four rows together;
// with a workgroup, wave w adds row w's, the waves' sums meet in LDS, and wave w adds the
// total of row w to C.  A row is in no other work item: no atomics.
template <typename T, int TN, int EDGE, int WPG>
__global__ void __launch_bounds__(kWgThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
spmm_group_kernel(int n, int n_groups, const RowGroup* __restrict__ groups, const int* __restrict__ row_ptr,
                  const int* __restrict__ col, const typename DenseVec<T>::Acc* __restrict__ val,
                  const T* __restrict__ B, typename DenseVec<T>::Acc* __restrict__ C, bool overwrite)
{
    using S = SpmmShape<T, TN>;
    using A = typename S::Acc;
    constexpr int VEC = S::kVec, LPR = S::kLpr, G = S::kGroupsWave, R = kGroupRows;
    constexpr int GPW = kWavesPerWg / WPG; // groups per workgroup
    static_assert(WPG == 1 || WPG == kWavesPerWg, "a group has one wave, or one workgroup");
    __shared__ __attribute__((aligned(16))) int lds_c[kWavesPerWg][WPG == 1 ? R : 1][kWave];
    __shared__ __attribute__((aligned(16))) A lds_v[kWavesPerWg][R][kWave];
    __shared__ __attribute__((aligned(16))) A sums[WPG > 1 ? kWavesPerWg : 1][R][TN];
    // (the wave's number is the same in all its lanes; saying so keeps the group's description,
    // the position in the run and the addresses of its dense rows in scalar registers)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int g = xcd_logical_block(blockIdx.x, gridDim.x) * GPW + wave / WPG;
    if (g >= n_groups) return;
    if (groups[g].len <= 0) return; // not a group: its rows are in the lists
    const RowGroup d = shared_run(groups[g]); // the columns [lo, lo + len) that all four runs hold
    const int w = wave % WPG; // this wave among the waves of its group
    const int ls = lane % LPR, group = lane / LPR;
    const int tile = blockIdx.y * TN;
    const bool col_ok = !EDGE || tile + ls * VEC < n;
    const T* b_lane = B + tile + (col_ok ? ls * VEC : 0);
    const int row0 = g * R;
    // per row: the slot of column j of the shared run is at[r] + j
    int at[R];
#pragma unroll
    for (int r = 0; r < R; ++r) at[r] = row_ptr[row0 + r] + d.pos[r];

    // this wave's share of the run, in quads of columns
    const int quads = (d.len + 3) / 4;
    const int q_begin = quads * w / WPG, q_end = quads * (w + 1) / WPG;
    const int j_end = min(d.len, 4 * q_end);
    A acc[R][VEC];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int x = 0; x < VEC; ++x) acc[r][x] = A(0);
    // a dense row of the run = a scalar address (start of the run, step, quad) + this lane's
    // 32-bit offset (its lane group's quad, its elements of the tile, the row in the quad)
    const T* b_run = B + tile + (size_t)d.lo * n;
    const unsigned row_bytes = (unsigned)n * (unsigned)sizeof(T);
    const unsigned lane_off = 4u * group * row_bytes + (col_ok ? ls * VEC * (unsigned)sizeof(T) : 0u); // in bytes
    A v_next[R]; // the values of the next step are loaded while this one is computed
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = 4 * q_begin + lane;
        v_next[r] = j < j_end ? val[at[r] + j] : A(0);
    }
    for (int j0 = 4 * q_begin; j0 < j_end; j0 += kWave) {
#pragma unroll
        for (int r = 0; r < R; ++r) lds_v[wave][r][lane] = v_next[r];
        wave_lds_sync();
        {
            const int j = j0 + kWave + lane;
#pragma unroll
            for (int r = 0; r < R; ++r) v_next[r] = j < j_end ? val[at[r] + j] : A(0);
        }
        const int nq = min(kWave / 4, (j_end - j0 + 3) / 4);
#pragma unroll
        for (int i = 0; i < kWave / 4 / G; ++i) {
            const int q = group + i * G;
            if (q < nq) {
                // four consecutive rows of B (the last quad of a run may be cut short: its rows
                // past the run repeat the run's last row, which every row of the group
                // references; their values are zero)
                const char* b_quad = reinterpret_cast<const char*>(b_run + (size_t)(j0 + 4 * i * G) * n);
                const int room = d.len - 1 - (j0 + 4 * q);
                const unsigned o1 = room >= 1 ? row_bytes : 0u;
                const unsigned o2 = room >= 2 ? 2u * row_bytes : o1;
                const unsigned o3 = room >= 3 ? 3u * row_bytes : o2;
                const unsigned off[4] = {lane_off, lane_off + o1, lane_off + o2, lane_off + o3};
                A b[4][VEC];
#pragma unroll
                for (int t = 0; t < 4; ++t) DenseVec<T>::load(reinterpret_cast<const T*>(b_quad + off[t]), b[t]);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    A v[4];
                    load_quad(&lds_v[wave][r][4 * q], v);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int x = 0; x < VEC; ++x) acc[r][x] = fma(v[t], b[t][x], acc[r][x]);
                }
            }
        }
        wave_lds_sync();
    }
    if constexpr (WPG == 1) {
        // the nonzeros outside the run, of the four rows at once: their columns and values are
        // loaded together and their gathers follow each other without a wait in between (row
        // after row, a wave would sit through two memory round trips per row and step)
        int row_first[R], split[R], jump[R], cnt[R], max_cnt = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            row_first[r] = at[r] - d.pos[r];
            split[r] = d.pos[r];
            jump[r] = d.len;
            cnt[r] = split[r] + (row_ptr[row0 + r + 1] - (at[r] + d.len)); // the slots before the run + those after it
            max_cnt = max(max_cnt, cnt[r]);
        }
        for (int off = 0; off < max_cnt; off += kWave) {
            const int slot = off + lane;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int live = min(cnt[r] - off, kWave); // this row's slots in this step (may be <= 0)
                int c = 0;
                A v = A(0);
                if (lane < ((live + 3) & ~3)) { // (slots past the end of the last quad: value 0, column of a real slot)
                    const bool past = slot >= cnt[r];
                    const int slot_at = past ? cnt[r] - 1 : slot;
                    const int idx = row_first[r] + slot_at + (slot_at >= split[r] ? jump[r] : 0);
                    c = col[idx];
                    v = past ? A(0) : val[idx];
                }
                lds_c[wave][r][lane] = c;
                lds_v[wave][r][lane] = v;
            }
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int live = min(cnt[r] - off, kWave);
                if (live >= kWave)
                    spmm_gather<T, TN, 16 / G, true>(b_lane, (size_t)n, acc[r], lds_c[wave][r], lds_v[wave][r], group, G, 16);
                else if (live > 0)
                    spmm_gather<T, TN, 16 / G, false>(b_lane, (size_t)n, acc[r], lds_c[wave][r], lds_v[wave][r], group, G,
                                                      (live + 3) / 4);
            }
            wave_lds_sync();
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int x = 0; x < VEC; ++x) acc[r][x] = butterfly_sum<LPR, kWave>(acc[r][x]);
            if (group == 0 && col_ok) {
                A* c_lane = C + (size_t)(row0 + r) * n + tile + ls * VEC;
#pragma unroll
                for (int x = 0; x < VEC; ++x) c_lane[x] = overwrite ? acc[r][x] : c_lane[x] + acc[r][x]; // (added by contract, unless told to store)
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int x = 0; x < VEC; ++x) acc[r][x] = butterfly_sum<LPR, kWave>(acc[r][x]);
            if (group == 0) {
#pragma unroll
                for (int x = 0; x < VEC; ++x) sums[wave][r][ls * VEC + x] = acc[r][x];
            }
        }
        __syncthreads();
        // the row this wave finishes: its nonzeros before and after the run, then the update of C
#pragma unroll
        for (int r = w; r < R; r += WPG) {
            const int row = row0 + r, s = row_ptr[row], e = row_ptr[row + 1];
            const int run_first = s + d.pos[r], run_end = run_first + d.run(r);
            A outside[VEC]; // the slots before the run and, in the same pass, those after it
            spmm_sum_slots<T, TN>(s, 0, (run_first - s) + (e - run_end), run_first - s, d.run(r), lane, lds_c[wave][0],
                                  &lds_v[wave][0][0], b_lane, n, col, val, outside);
            if (group == 0 && col_ok) {
                A* c_lane = C + (size_t)row * n + tile + ls * VEC;
#pragma unroll
                for (int x = 0; x < VEC; ++x) {
                    A total = outside[x];
#pragma unroll
                    for (int v = 0; v < WPG; ++v) total += sums[v][r][ls * VEC + x];
                    c_lane[x] = overwrite ? total : c_lane[x] + total; // (added by contract, unless told to store)
                }
            }
        }
    }
}

// The rows of a hub plan, cut into pieces by column slab (rode_items.hpp), slab after slab, so that the hub rows' nonzeros of
// one slab of B are worked on at the same time on one XCD and find B's rows in its L2.  A piece's sum goes to its own row
// of `partial` (piece = slab group * hub rows + hub row; spmm_hub_reduce_kernel adds a row's
// pieces up), or, without that workspace, is added to its row of C atomically (a hub row
// then gets one atomic row update per slab: slower than the plain kernels at 512-byte rows).
// A piece that waves share is finished by the wave that has its first step.
template <typename T, int TN, int EDGE>
__global__ void __launch_bounds__(kHubWavesMax * kWave)
spmm_hub_kernel(int n, HubGrid grid, const int* __restrict__ hub, const int* __restrict__ col,
                const typename DenseVec<T>::Acc* __restrict__ val, const T* __restrict__ B,
                typename DenseVec<T>::Acc* __restrict__ C, typename DenseVec<T>::Acc* __restrict__ partial)
{
    using S = SpmmShape<T, TN>;
    using A = typename S::Acc;
    constexpr int VEC = S::kVec, LPR = S::kLpr, G = S::kGroupsWave;
    __shared__ __attribute__((aligned(16))) int lds_c[kHubWavesMax * kWave];
    __shared__ __attribute__((aligned(16))) A lds_v[kHubWavesMax * kWave];
    __shared__ __attribute__((aligned(16))) A heads[kHubWavesMax][TN]; // a wave's sum of a piece that an earlier wave began
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave; // (uniform: scalar registers)
    const HubPlan hp = hub_plan_view(hub);
    const int wg = xcd_logical_block(blockIdx.x, gridDim.x);
    int steps;
    const HubShare share = hub_share(hp, grid, wg, wave, lane, steps);
    const int ls = lane % LPR, group = lane / LPR;
    const int tile = blockIdx.y * TN;
    const bool col_ok = !EDGE || tile + ls * VEC < n;
    const T* b_lane = B + tile + (col_ok ? ls * VEC : 0);
    constexpr int EPG = VEC / G > 0 ? VEC / G : 1; // elements each group adds
    A total[VEC];
    int open = -1; // the piece that `total` is the first part of
    for (unsigned long long todo = share.pieces; todo; todo &= todo - 1ull) {
        const int i = __builtin_ctzll(todo);
        const HubPart p = hub_part(share, i);
        spmm_sum_slots<T, TN, 0, kInEights<EDGE>>(p.base, 0, p.cnt, p.cnt, 0, lane, lds_c + wave * kWave, lds_v + wave * kWave, b_lane, n, col, val, total);
        if (!partial) {
            A* c_lane = C + (size_t)p.row * n + tile + ls * VEC;
#pragma unroll
            for (int x = 0; x < VEC; ++x)
                if (group == x / EPG && col_ok) atomicAdd(c_lane + x, total[x]);
        } else if (!p.starts) {
            if (group == 0) {
#pragma unroll
                for (int x = 0; x < VEC; ++x) heads[wave][ls * VEC + x] = total[x];
            }
        } else if (p.ends) {
            if (group == 0 && col_ok) store_row<VEC>(partial + ((size_t)wg * grid.pieces + i) * n + tile + ls * VEC, total);
        } else {
            open = i; // (the last of this wave's pieces)
        }
    }
    if (!partial) return;
    __syncthreads();
    if (open >= 0) {
        const int end = __builtin_amdgcn_readlane(share.before, open) + __builtin_amdgcn_readlane(share.steps, open);
        for (int w = wave + 1; w < grid.waves && hub_first_step(grid, steps, w) < end; ++w) {
            if (hub_first_step(grid, steps, w) == hub_first_step(grid, steps, w + 1)) continue; // (fewer steps than waves: it has none)
#pragma unroll
            for (int x = 0; x < VEC; ++x) total[x] += heads[w][ls * VEC + x];
        }
        if (group == 0 && col_ok) store_row<VEC>(partial + ((size_t)wg * grid.pieces + open) * n + tile + ls * VEC, total);
    }
}

// C[hub row, :] += sum of the row's pieces (a hub row is in no other work item, so no
// atomics; added, not stored, because long rows are accumulated into C by contract).  One workgroup per hub row: a group of n * sizeof / 16 threads reads a
// piece's partial row 16 bytes per thread, the groups take the slabs in turn and their
// sums are added up through LDS in a fixed order.
template <typename A>
__global__ void __launch_bounds__(kWgThreads)
spmm_hub_reduce_kernel(int n, HubGrid grid, const int* __restrict__ hub, const A* __restrict__ partial, A* __restrict__ C)
{
    constexpr int V = 16 / sizeof(A);
    __shared__ __attribute__((aligned(16))) A sums[kWgThreads * V];
    const HubPlan hp = hub_plan_view(hub);
    const int merge = grid.merge, i = blockIdx.x;
    if (i >= grid.rows) return;
    const int h = grid.longs ? hp.longs[i] : i;
    const int* piece = hp.pieces + (size_t)h * (hp.slabs + 1);
    A* c_row = C + (size_t)hp.rows[h] * n;
    const int vecs = n / V; // 16-byte pieces of a row (n * sizeof(A) is a multiple of 16)
    for (int v0 = 0; v0 < vecs; v0 += kWgThreads) {
        const int width = min(vecs - v0, kWgThreads); // threads side by side on one partial row
        const int groups = kWgThreads / width;
        const int group = threadIdx.x / width, v = v0 + threadIdx.x % width;
        A sum[V];
#pragma unroll
        for (int x = 0; x < V; ++x) sum[x] = A(0);
        if (group < groups) {
            for (int sg = group; sg * merge < hp.slabs; sg += groups) {
                if (piece[min(sg * merge + merge, hp.slabs)] > piece[sg * merge]) {
                    const A* src = partial + ((size_t)sg * grid.rows + i) * n + (size_t)v * V;
#pragma unroll
                    for (int x = 0; x < V; ++x) sum[x] += src[x];
                }
            }
        }
#pragma unroll
        for (int x = 0; x < V; ++x) sums[threadIdx.x * V + x] = sum[x];
        __syncthreads();
        if (group == 0) {
            for (int g = 1; g < groups; ++g) {
#pragma unroll
                for (int x = 0; x < V; ++x) sum[x] += sums[(g * width + threadIdx.x) * V + x];
            }
#pragma unroll
            for (int x = 0; x < V; ++x) c_row[(size_t)v * V + x] += sum[x];
        }
        __syncthreads();
    }
}

constexpr int kClearRowsPerGroup = 8;

// Zeroes exactly the rows of C that the two SpMM kernels do not overwrite: rows whose
// aligned length N = len + (start & 3) is >= 32 are accumulated into (but, under
// kSpmmOverwrite, those of at most `stored` slots: spmm_overwrite_limit), rows with N == 0
// belong to no work item; rows with 0 < N < 32 are stored by the residue kernel and
// are left alone.  16 lanes x 16 bytes per step and row.
__global__ void __launch_bounds__(kWgThreads)
spmm_clear_rows_kernel(int M, size_t row_bytes, int stored, const int* __restrict__ row_ptr, char* __restrict__ C)
{
    constexpr int kLanes = 16, kGroups = kWgThreads / kLanes;
    const int group = threadIdx.x / kLanes, lane = threadIdx.x % kLanes;
    const int first = xcd_logical_block(blockIdx.x, gridDim.x) * (kGroups * kClearRowsPerGroup);
    // batch b of a workgroup covers kGroups consecutive rows, one per lane group
    int s[kClearRowsPerGroup], e[kClearRowsPerGroup];
#pragma unroll
    for (int b = 0; b < kClearRowsPerGroup; ++b) {
        const int row = first + b * kGroups + group;
        s[b] = row < M ? row_ptr[row] : 1;
        e[b] = row < M ? row_ptr[row + 1] : 2; // N = 2: a row that is left alone
    }
#pragma unroll
    for (int b = 0; b < kClearRowsPerGroup; ++b) {
        const int N = e[b] - s[b] + (s[b] & (kVecLen - 1));
        if (N > 0 && (N < kBlockItems || N <= stored)) continue;
        char* dst = C + (size_t)(first + b * kGroups + group) * row_bytes;
        for (size_t off = lane * 16; off < row_bytes; off += kLanes * 16)
            *reinterpret_cast<uint4*>(dst + off) = make_uint4(0, 0, 0, 0);
    }
}

inline int grid_for_waves(long long nwaves)
{
    long long wgs = (nwaves + kWavesPerWg - 1) / kWavesPerWg;
    wgs = (wgs + kXcds - 1) / kXcds * kXcds; // xcd_logical_block needs a multiple of kXcds
    // a launch dimension holds fewer than 2^32 threads; more work items than that (over
    // 16 M workgroups) are refused instead of being launched wrongly
    return wgs * kWgThreads < (1ll << 32) ? (int)wgs : -1;
}

inline HubRows spmm_hub_rows(const int* counts, int n, int tile, size_t elem)
{
    return hub_rows_of_call(counts, n * elem, tile * elem, (n + tile - 1) / tile, 18, 600, (size_t)8 * kHubSlabRows * counts[1]);
}

template <typename T, int TN, int EDGE>
hipError_t launch(int m1, int m2, int n, const int* block_rows, const int* residue_rows, const int* st_off,
                  const int* row_ptr, const int* col, const typename DenseVec<T>::Acc* val, const T* B,
                  typename DenseVec<T>::Acc* C, int flags, PlanRef plan, hipStream_t s1, hipStream_t s2)
{
    const int tiles = (n + TN - 1) / TN;
    // a usable hub plan takes its rows out of both lists (the caller promised whole lists with it)
    const bool hub_plan = plan.hub != nullptr && plan.hub_counts != nullptr && plan.hub_counts[3] != 0 &&
                          plan.hub_counts[0] > 0;
    const HubRows hub_rows = hub_plan ? spmm_hub_rows(plan.hub_counts, n, TN, sizeof(T)) : HubRows();
    // (rows known to be short: one wave has no more to do for all of a row)
    const bool short_rows = plan.longest > 0 && plan.longest <= kShortRowSlots && !hub_plan;
    const int owned_slots = (flags & kSpmmWholeLists) && (m1 >= kOwnedMinSegments || short_rows) ? kOwnedRowSlots : 0;
    // what the block kernel is told: rows it owns, or (negative) only that it may merge short
    // segments - which needs no promise, and with this many segments costs no parallelism
    const int block_owned = owned_slots > 0 ? owned_slots : (m1 >= kMergeMinSegments ? -1 : 0);
    const bool group_plan = plan.groups != nullptr && plan.group_counts != nullptr && plan.group_counts[1] > 0;
    RowOwners owners;
    owners.hub_min_len = hub_rows.min_len;
    if (group_plan) {
        owners.groups = reinterpret_cast<const RowGroup*>(plan.groups + kGroupHeaderInts);
        owners.n_groups = plan.group_counts[0];
    }
    // rows with a single work item are stored instead of added (spmm_overwrite_limit says which)
    const bool overwrite = (flags & kSpmmOverwrite) != 0;
    owners.overwrite = overwrite && owned_slots > 0 && !hub_plan;
    const bool in_parts = short_rows && m1 < kOwnedMinSegments && owners.overwrite;
    const int only = flags & kOnlyMask; // one kernel family of the call (timing each on its own)
    const bool hubs = hub_rows.rows > 0 && (only == 0 || only == kSpmmOnlyHub);
    const bool grouped = group_plan && (only == 0 || only == kSpmmOnlyHub); // (timed with the hub kernels)
    constexpr int RPW = kWave / SpmmShape<T, TN>::kLpr;
    const int shards = plan.shards > 1 ? plan.shards : 1, tile_rows = plan.shards > 1 ? 1 : tiles;
    // (segments per wave: known only when the caller said how long its segments are and merging is on.
    // A sharded launch has a wave per segment and tile: with many of them a wave takes several rows - 16 K
    // rows of 40 nonzeros, width 128: 41 -> 32 us - later than an unsharded one, as long rows need the waves)
    const int walked = shards > 1 ? (int)min((long long)m1 * shards / 3, (long long)INT32_MAX) : m1;
    const int chunk_hint = block_owned != 0 ? chunk_for_segments(plan.seg_length, walked) : (plan.seg_length > 0 ? 1 : 0);
    const int g1 = chunk_hint > 0 ? grid_for_waves((m1 + chunk_hint - 1) / chunk_hint) : grid_for_waves(min(m1, kBlockGridWaves));
    const int g2 = grid_for_waves(((long long)m2 + RPW - 1) / RPW);
    if (g1 < 0 || g2 < 0 || tiles > 65535) return hipErrorInvalidConfiguration;
    if ((long long)max(g1, g2) * shards * kWgThreads >= (1ll << 32)) return hipErrorInvalidConfiguration;
    // With a host copy of the plan's header, a kernel that would find every chunk taken by
    // the other one is not launched at all.
    bool standard_residue = true, window_residue = plan.dev != nullptr;
    if (plan.dev && plan.host_counts) {
        standard_residue = plan.host_counts[1] < plan.host_counts[0];
        window_residue = plan.host_counts[1] > 0;
    }
    // (every row in a group with a run: the lists' kernels would find nothing to do)
    const bool lists = !(group_plan && plan.group_counts[2] == 0);
    const bool block = lists && m1 > 0 && (only == 0 || only == kSpmmOnlyBlock);
    const bool residue = lists && m2 > 0 && (only == 0 || only == kSpmmOnlyResidue);
    hipError_t e = hipSuccess;
    // (without block segments only where C is not cleared and the launch is small: the residue kernel has more waves per CU)
    const bool alone = m1 == 0 && plan.c_rows > 0 && short_rows && (long long)g2 * tiles <= kPairMaxAlone;
    const bool pair = (block || alone) && residue && standard_residue && s1 == s2 &&
                      (long long)(g1 + g2) * tiles <= (shards > 1 ? kPairMaxSharded : kPairMaxWorkgroups);
    int g0 = 0;
    bool wide = false;
    if (plan.c_rows > 0) { // C is not cleared
        const bool all_stored = pair && owners.overwrite && !group_plan && plan.dev == nullptr && plan.longest > 0;
        wide = all_stored && chunk_hint == 1 && plan.longest > kOwnedRowSlots && wide_rows_pay(plan.longest, plan.seg_length, TN * sizeof(T), (size_t)plan.nonzeros * n * sizeof(T), EDGE != 0);
        if (wide || (all_stored && plan.longest <= kOwnedRowSlots)) {
            g0 = empty_row_workgroups(plan.c_rows);
        } else {
            e = spmm_clear_rows_launch(plan.c_rows, (size_t)n * sizeof(typename DenseVec<T>::Acc), owners.overwrite ? kOwnedRowSlots : 0, row_ptr, C, s1);
            if (e != hipSuccess) return e;
        }
    }
    if (pair) {
        dim3 grid((g0 + g1 + g2) * shards, tile_rows);
        auto kernel = owners.overwrite ? spmm_pair_kernel<T, TN, EDGE, 2, true> : spmm_pair_kernel<T, TN, EDGE, 2, false>;
        if (in_parts)
            kernel = spmm_pair_kernel<T, TN, EDGE, 3, true>;
        else if (wide)
            kernel = spmm_pair_kernel<T, TN, EDGE, 4, true>;
        else if (chunk_hint == 1)
            kernel = owners.overwrite ? spmm_pair_kernel<T, TN, EDGE, 0, true> : spmm_pair_kernel<T, TN, EDGE, 0, false>;
        else if (chunk_hint > 1)
            kernel = owners.overwrite ? spmm_pair_kernel<T, TN, EDGE, 1, true> : spmm_pair_kernel<T, TN, EDGE, 1, false>;
        kernel<<<grid, kWgThreads, 0, s1>>>(shards, g0, plan.c_rows, g1, m1, m2, n, block_owned, chunk_hint, owners, block_rows, residue_rows, st_off,
                                            row_ptr, col, val, B, C, plan.dev);
        e = hipGetLastError();
    } else {
        if (block) {
            dim3 grid(g1 * shards, tile_rows);
            auto kernel = spmm_block_kernel<T, TN, EDGE, 2, false>;
            if (in_parts)
                kernel = spmm_block_kernel<T, TN, EDGE, 3, true>;
            else if (chunk_hint == 1)
                kernel = owners.overwrite ? spmm_block_kernel<T, TN, EDGE, 0, true> : spmm_block_kernel<T, TN, EDGE, 0, false>;
            else if (chunk_hint > 1)
                kernel = owners.overwrite ? spmm_block_kernel<T, TN, EDGE, 1, true> : spmm_block_kernel<T, TN, EDGE, 1, false>;
            else if (owners.overwrite)
                kernel = spmm_block_kernel<T, TN, EDGE, 2, true>;
            kernel<<<grid, kWgThreads, 0, s1>>>(shards, m1, n, block_owned, chunk_hint, owners, block_rows, st_off, row_ptr, col, val, B, C);
            e = hipGetLastError();
        }
        if (residue && standard_residue) {
            dim3 grid(g2 * shards, tile_rows);
            spmm_residue_kernel<T, TN, (EDGE != 0 ? kPartial : 0)><<<grid, kWgThreads, 0, s2>>>(shards, m2, n, owned_slots, owners, residue_rows, row_ptr, col,
                                                                          val, B, C, plan.dev);
            if (e == hipSuccess) e = hipGetLastError();
        }
    }
    if (e == hipSuccess && hubs) {
        using A = typename DenseVec<T>::Acc;
        const long long pieces = (long long)hub_rows.rows * hub_groups(plan.hub_counts[1], hub_rows.merge);
        const HubGrid hub_wgs = hub_grid(hub_rows, plan.hub_counts[1]);
        if (hub_wgs.wgs < 0) return hipErrorInvalidConfiguration;
        dim3 grid(hub_wgs.wgs, tiles);
        const size_t need = (size_t)pieces * n * sizeof(A);
        A* partial = plan.hub_workspace && plan.hub_workspace_bytes >= need ? static_cast<A*>(plan.hub_workspace) : nullptr;
        spmm_hub_kernel<T, TN, EDGE><<<grid, hub_wgs.waves * kWave, 0, s1>>>(n, hub_wgs, plan.hub, col, val, B, C, partial);
        if (partial) spmm_hub_reduce_kernel<A><<<hub_rows.rows, kWgThreads, 0, s1>>>(n, hub_wgs, plan.hub, partial, C);
        e = hipGetLastError();
    }
    if (e == hipSuccess && grouped) {
        // one wave per group when there are groups enough to fill the GPU that way (measured on
        // the attention-mask benchmark, 4096 groups: 0.042 against 0.062 ms), else a workgroup
        if (plan.group_counts[1] >= kGroupWaveEach) {
            const int wgs = (owners.n_groups + kWavesPerWg - 1) / kWavesPerWg;
            dim3 grid((wgs + kXcds - 1) / kXcds * kXcds, tiles);
            spmm_group_kernel<T, TN, (EDGE != 0 ? kPartial : 0), 1><<<grid, kWgThreads, 0, s1>>>(n, owners.n_groups, owners.groups, row_ptr, col,
                                                                           val, B, C, overwrite);
        } else {
            dim3 grid((owners.n_groups + kXcds - 1) / kXcds * kXcds, tiles);
            spmm_group_kernel<T, TN, (EDGE != 0 ? kPartial : 0), kWavesPerWg><<<grid, kWgThreads, 0, s1>>>(n, owners.n_groups, owners.groups, row_ptr,
                                                                                     col, val, B, C, overwrite);
        }
        e = hipGetLastError();
    }
    if (e == hipSuccess && residue && window_residue)
        e = spmm_window_launch<T>(m2, n, owned_slots, col, val, B, C, plan, s2);
    return e;
}

template <typename T, int TN>
hipError_t launch_edge(int m1, int m2, int n, const int* block_rows, const int* residue_rows, const int* st_off,
                       const int* row_ptr, const int* col, const typename DenseVec<T>::Acc* val, const T* B,
                       typename DenseVec<T>::Acc* C, int flags, PlanRef plan, hipStream_t s1, hipStream_t s2)
{
    if constexpr (TN >= 64 && sizeof(T) <= 4)
        if (n % TN && n % 32 == 0) // (spmm_tile_of_call)
            return launch<T, TN, kPartialEights>(m1, m2, n, block_rows, residue_rows, st_off, row_ptr, col, val, B, C, flags, plan, s1, s2);
    return n % TN ? launch<T, TN, kPartial>(m1, m2, n, block_rows, residue_rows, st_off, row_ptr, col, val, B, C,
                                            flags, plan, s1, s2)
                  : launch<T, TN, 0>(m1, m2, n, block_rows, residue_rows, st_off, row_ptr, col, val, B, C,
                                     flags, plan, s1, s2);
}

} // namespace

// The longest row (in aligned slots) that an SpMM call with m1 block segments, the whole-lists
// promise and kSpmmOverwrite stores with a single work item instead of adding to it; 0: none
// of the rows that have block segments (rows of fewer than 32 aligned slots are always
// stored, rows of kept groups of a group plan under kSpmmOverwrite as well).
int spmm_overwrite_limit(int m1, bool hub_plan) { return m1 >= kOwnedMinSegments && !hub_plan ? kOwnedRowSlots : 0; }

// The dense row is cut into tiles of 32, 64 or 128 columns (at most 32 lanes of 16 bytes per tile row);
// the tile width with the least padding wins, the widest on a tie.
static int spmm_tile_width(int n, size_t elem)
{
    auto padded = [n](int tn) { return (n + tn - 1) / tn * tn; };
    int best = 32;
    if (padded(64) <= padded(best)) best = 64;
    if (elem <= 4 && padded(128) <= padded(best)) best = 128;
    return best;
}

// ... but for some calls whose least padding is with tiles of 32 columns (widths like 96, 160, 224).  us of 32 / 64 / 128 columns, uniform (u)
// and lognormal degrees, two matrices in turn:
// Halves: a tile of 32 is half a line of 128 bytes, which is fetched for each of the two.  Tiles of 128 (u 16 K of 110 x 96 34.6 / 29.4 / 24.1, 60 K of 20
// 51 / 44 / 37, 400 K of 14 336 / 279 / 218), but of 64
//   * where those of 128 have a quarter of their lanes and more idle, up to 30 MB (x 160: u 33 K of 110 120 / 119 / 144; 48 MB and more 1 / 0.80 to
//     0.89 / 0.73 to 0.86);
//   * where the dense operand is near the size of an L2 and its rows are used less than 12 times (u 33 K of 8 x 96 13.3 / 13.4 / 14.7), up to 3.5 MB
//     less than 24 (16.5 K of 20 x 96 9.9 / 9.4 / 10.6); less than 10 times and 12 to 16 MB, those of 32 (u 33 K of 8 x 224 22.8 / 25.6 / 24.9);
//   * where one wave has all of a row, and the wider its tiles the longer for it, up to 1024 slots at 1 to 2.5 ns: 128 columns from 200 KB to
//     gather for each of its slots on, 64 from 90 KB (x 96: 12 K of 14, 899 slots, 36 KB each 11.4 / 14.5 / 16.3; 20 K of 20, 72 KB 18.9 / 17.4 / 20.2;
//     26 K of 32, 155 KB 32 / 27 / 30; 60 K of 14, 156 KB 38 / 34 / 33; 60 K of 32, 360 KB 74 / 70 / 60).
//     Rows of equal length have no such row, if they are more than tails (u x 96, 1 / 128 columns: 4000 of 30 0.81, of 60 0.72, 12 K of 60 0.68, 30 K of 22
//     0.77, but 4000 of 8 to 22 1.13 to 1.20).
//   * Both are otherwise with rows of unequal length and an operand past the L2s, which is waited for longer than that row: from 60 KB on, and near the
//     size of an L2 as well (lognormal x 96: 30 K of 8, 42 KB 15.6 / - / 19.1, 30 K of 22, 124 KB 28.2 / 26.1 / 24.1, 60 K of 8, 90 KB 27.1 / 27.1 / 24.1, 100 K of
//     8 44.0 / 41.8 / 36.5).
// 32-bit operands: one line at a time keeps more of the operand in the L2s, as long as its tiles fit at all (sharding_pays); below 2.5 MB and above
// 26 MB a tile whole rows are better, if a quarter of the lanes at most has nothing and with 500 KB to gather for each slot of the longest row
// (u 4000 of 40 x 96 9.9 -> 8.2, 230 K of 12 167 -> 161, 300 K of 10 187 -> 178, between them u 10 K of 20 8.2 -> 9.0, u 16 K of 110 37 -> 43; 4000 of 32,
// 1024 slots, 48 KB 8.4 -> 15.2).
// Where neighbouring rows' columns lie close together the halves of a line meet in the caches anyway (halves, a band of 128, width 96: 70 K of 12
// 11.9 -> 12.5, but 200 K of 20 55.9 -> 46.7).
static int spmm_tile_of_call(int n, size_t elem, const PlanRef& plan)
{
    const int least = spmm_tile_width(n, elem);
    // (a group's four rows have no registers for sums of eight)
    if (least != 32 || n <= 32 || elem > 4 || n % 32 != 0 || plan.groups) return least;
    constexpr size_t KB = 1000, MB = 1000000;
    const size_t rows = plan.dense_rows, nonzeros = plan.nonzeros, bytes = rows * n * elem, gathered = nonzeros * n * elem;
    size_t slots = plan.longest > 0 && plan.longest < kOwnedRowSlots ? plan.longest : kOwnedRowSlots;
    if (plan.equal_rows >= (bytes < 5 * MB ? 28 : 16)) slots = min(slots, (size_t)2 * plan.equal_rows); // (not said in calls whose rows are all stored)
    auto enough = [&](size_t each) { return nonzeros == 0 || gathered >= slots * each; }; // (not said: taken to be)
    if (plan.columns_local && bytes < 26 * MB) return 32;
    const bool filled = 3 * ((n + 127) / 128 * 128) <= 4 * n;
    if (elem == 4) return filled && rows > 0 && (bytes <= 5 * MB / 2 || rows * 128 > 27 * MB) && enough(500 * KB) ? 128 : 32;
    const bool ragged = plan.equal_rows == 0 && bytes >= 11 * MB / 2;
    if (!ragged && nonzeros > 0 && nonzeros < 10 * rows && bytes > 12 * MB && bytes < 16 * MB) return 32;
    const bool near_l2 = !ragged && nonzeros > 0 && nonzeros < (bytes < 7 * MB / 2 ? 24 : 12) * rows && bytes >= 3 * MB && bytes <= 12 * MB;
    return (filled || bytes >= 30 * MB) && !near_l2 && enough((ragged ? 60 : 200) * KB) ? 128 : enough((ragged ? 60 : 90) * KB) ? 64 : 32;
}

// The partial rows that the hub kernels of an SpMM of this width want, for operands of 4 (or, if more, 2) or of 8 bytes an element.
size_t spmm_hub_partial_rows(const int* counts, int n, int acc_bytes)
{
    size_t most = 0;
    for (size_t elem = acc_bytes; elem >= (acc_bytes == 8 ? 8 : 2); elem /= 2) {
        for (int tile = 32; tile <= (elem > 4 ? 64 : 128); tile *= 2) { // (any that a call of this width may take)
            if (tile != spmm_tile_width(n, elem) && (n % 32 != 0 || spmm_tile_width(n, elem) != 32 || n == 32)) continue;
            const HubRows use = spmm_hub_rows(counts, n, tile, elem);
            const size_t rows = (size_t)use.rows * hub_groups(counts[1], use.merge);
            most = rows > most ? rows : most;
        }
    }
    return most;
}

// n: any positive multiple of the 128-bit vector width (4 fp32, 8 fp16, 2 fp64).  Multiples of 32 (all
// the reference supports) run without any bounds test.  Chunks of the residue list for
// which `plan` holds a window go to the ring or window kernel, of those that take the
// width (ring_slices, window_takes), where that pays (choose_windows).
template <typename T>
hipError_t spmm_launch(int m1, int m2, int n, const int* block_rows, const int* residue_rows, const int* st_off,
                       const int* row_ptr, const int* col, const typename SpmmAcc<T>::type* val, const T* B,
                       typename SpmmAcc<T>::type* C, int flags, PlanRef plan, hipStream_t s1, hipStream_t s2)
{
    static_assert(std::is_same<typename SpmmAcc<T>::type, typename DenseVec<T>::Acc>::value, "accumulation type");
    if (n <= 0 || n % DenseVec<T>::kElems != 0) return hipErrorInvalidValue;
    constexpr WindowGain kWide = {0.87f, 0.0237f, 1.17f, 300, 1.17f, 300}, kNarrow = {0.715f, 0.0235f, 1.f, 380, 1.17f, 380},
                         kHalves = {0.79f, 0.0113f, 1.07f, 270, 1.17f, 380}, kDoubles = {0.75f, 0.0228f, 1.f, 360, 1.17f, 360};
    const size_t row_bytes = (size_t)n * sizeof(T);
    const int slices = ring_slices(row_bytes);
    // (a band of 128 columns is worth 5 % less than those of 192 and 256 that the figures beside rings_pay are of)
    const bool line = row_bytes == 128, whole = slices == 1;
    const WindowGain ring = sizeof(T) == 8 ? WindowGain{line ? 1.2f : whole ? 0.94f : 1.1f, line ? 0.03f : whole ? 0.025f : 0.02f, 1.f, 0, 1.f, 0}
                            : sizeof(T) == 2 ? WindowGain{line ? 0.72f : whole ? 0.93f : 0.97f, line ? 0.0145f : 0.02f, 1.f, 0, 1.f, 0}
                                             : WindowGain{line ? 0.67f : whole ? 0.94f : 1.1f, line ? 0.0235f : whole ? 0.025f : 0.02f, 1.f, 0, 1.f, 0};
    choose_windows(plan, m2, kWindowWgs, slices, window_takes(row_bytes), row_bytes, ring,
                   sizeof(T) == 8 ? kDoubles : sizeof(T) == 2 ? kHalves : row_bytes > 256 ? kWide : kNarrow);
    if constexpr (!std::is_same<T, double>::value) { // (a line of doubles is no tile width)
        constexpr int kLine = 128 / (int)sizeof(T);
        const int lines = n / kLine;
        // (a plan's kernels have their own ways to share dense rows)
        if (n % kLine == 0 && (lines == 2 || lines == 4 || lines == 8) && plan.dense_rows > 0 &&
            sharding_pays(lines, sizeof(T) == 2, plan.dense_rows, (long long)m1 + m2, 3ll * m1 > m2, plan.nonzeros) &&
            !plan.columns_local && plan.hub == nullptr && plan.groups == nullptr && plan.dev == nullptr) {
            plan.shards = lines;
            return launch<T, kLine, false>(m1, m2, n, block_rows, residue_rows, st_off, row_ptr, col, val, B, C, flags, plan, s1, s2);
        }
    }
    const int best = spmm_tile_of_call(n, sizeof(T), plan);
    if constexpr (sizeof(T) <= 4) {
        if (best == 128)
            return launch_edge<T, 128>(m1, m2, n, block_rows, residue_rows, st_off, row_ptr, col, val, B, C, flags,
                                       plan, s1, s2);
    }
    if (best == 64)
        return launch_edge<T, 64>(m1, m2, n, block_rows, residue_rows, st_off, row_ptr, col, val, B, C, flags, plan,
                                  s1, s2);
    return launch_edge<T, 32>(m1, m2, n, block_rows, residue_rows, st_off, row_ptr, col, val, B, C, flags, plan, s1, s2);
}

hipError_t spmm_clear_rows_launch(int M, size_t row_bytes, int stored, const int* row_ptr, void* C, hipStream_t stream)
{
    if (M <= 0) return hipSuccess;
    constexpr int kRowsPerWg = kWgThreads / 16 * kClearRowsPerGroup;
    long long wgs = ((long long)M + kRowsPerWg - 1) / kRowsPerWg;
    wgs = (wgs + kXcds - 1) / kXcds * kXcds;
    if (wgs * kWgThreads >= (1ll << 32)) return hipErrorInvalidConfiguration;
    spmm_clear_rows_kernel<<<(int)wgs, kWgThreads, 0, stream>>>(M, row_bytes, stored, row_ptr, static_cast<char*>(C));
    return hipGetLastError();
}

template hipError_t spmm_launch<float>(int, int, int, const int*, const int*, const int*, const int*, const int*,
                                       const float*, const float*, float*, int, PlanRef, hipStream_t, hipStream_t);
template hipError_t spmm_launch<__half>(int, int, int, const int*, const int*, const int*, const int*, const int*,
                                        const float*, const __half*, float*, int, PlanRef, hipStream_t, hipStream_t);
template hipError_t spmm_launch<double>(int, int, int, const int*, const int*, const int*, const int*, const int*,
                                        const double*, const double*, double*, int, PlanRef, hipStream_t, hipStream_t);

} // namespace rode
