// Launch functions behind the C ABI (one per kernel family).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stddef.h>

namespace rode {

size_t preprocess_workspace_bytes(int M);

// Largest matrix the allocation-free preprocessing entry point takes (RODE_HIP_STATIC_MAX_ROWS).
constexpr int kPreprocessStaticMaxRows = 4 * 1024 * 1024;
// Device address of the current GPU's static preprocessing scratch.
hipError_t preprocess_static_workspace(void** ptr);

hipError_t preprocess_launch(int seg, int kblock, int veclen, int M, const int* row_ptr, int* block_r_ind,
                             int* st_off, int* residue_r_ind, int* n_blk, int* n_res, void* workspace,
                             int capacity_blocks, hipStream_t stream, int plan_chunks = 0, int* plan_header = nullptr);
int preprocess_tile_rows(int M);
hipError_t preprocess_placed_launch(int seg, int kblock, int veclen, int M, const int* row_ptr, int* block_r_ind, int* st_off,
                                    int* residue_r_ind, int* n_blk, int* n_res, const unsigned long long* before, int capacity_blocks,
                                    int capacity_residue, hipStream_t stream, int plan_chunks, int* plan_header,
                                    const unsigned long long* places, int dense_rows, const int* col, int* windows);
bool preprocess_plan_too(int M); // does it take `places`?

// T = dense operand type; values, accumulators and C are float for T = float / __half
// and double for T = double.
template <typename T> struct SpmmAcc { using type = float; };
template <> struct SpmmAcc<double> { using type = double; };

// flags: the RODE_SPMM_* bits of the C ABI
constexpr int kSpmmWholeLists = 1, kSpmmOnlyBlock = 2, kSpmmOnlyResidue = 4, kSpmmOnlyHub = 8, kSpmmOverwrite = 16;
constexpr int kOnlyMask = kSpmmOnlyBlock | kSpmmOnlyResidue | kSpmmOnlyHub;

// A locality plan (rode_plan.hip): device array, and optionally a host copy of its four
// header ints (chunk counts), with which launches that have nothing to do are left out.
struct PlanRef {
    void no_window() { dev = nullptr, rows = nullptr, host_counts = nullptr; }
    const int* dev = nullptr;         // descriptors
    const void* rows = nullptr;       // planned rows of the chunks with a window
    const int* host_counts = nullptr;
    bool rings = false;               // the ring kernels take the chunks with a window (choose_windows)
    // A hub plan (rode_hub.hip) and the host copy of its eight header ints (required with it).
    const int* hub = nullptr;
    const int* hub_counts = nullptr;
    // SpMM only: room for one partial row of C per (slab, hub row), or null (atomics instead).
    void* hub_workspace = nullptr;
    size_t hub_workspace_bytes = 0;
    // A group plan (rode_group.hip) and the host copy of its four header ints (required with it).
    const int* groups = nullptr;
    const int* group_counts = nullptr;
    int tile_fours = 0;         // of its tiles (rode_hip_plans)
    // SDDMM: the RODE_SPMM_ONLY_* bits of the call (SpMM carries them in its flags)
    int only = 0;
    // SpMM: rows of the dense operand as the caller says (0: not said), and (set by spmm_launch) into how
    // many column tiles it is dealt out to the XCDs
    int dense_rows = 0, shards = 0;
    int nonzeros = 0;           // of the matrix, as the caller says (0: not said)
    // SpMM: rows of C where it is not cleared (0: it is, or every row is stored), the longest row in aligned slots (0: not said)
    int c_rows = 0, longest = 0;
    bool columns_local = false; // the caller knows that the columns of neighbouring rows lie close together
    int equal_rows = 0;         // nonzeros a row where no row has more than twice as many (0: not so, or not said)
    // Segment length of the decomposition the lists were made with, 0: not known
    int seg_length = 0;
};

// Do the window kernels pay for a call?  They take kWindowWgs chunks at a time, and a last round with few of them
// takes as long as a full one; against the standard kernels a full round gains the more, the more slots a row has
// (the window is copied either way).  full_round: that gain at s slots a row, base + per_slot * s, measured on bands of 128 to
// 256 in 130 K rows (1024 chunks); larger, largest: what becomes of it where the dense operands come near the size of the
// last-level cache (256 MB) and where they outgrow it (SDDMM: between the two the standard kernels still hit it, the copied windows
// no longer do; SpMM: the standard kernels lose it first).  us, standard -> window kernels, 9 / 14 / 18 / 27 slots:
//   SDDMM  f32 x 128    45 -> 32, 55 -> 36, 63 -> 38, 82 -> 44        1 M rows 358 -> 292, 458 -> 328, 544 -> 335, 740 -> 395
//          f32 x 64     24.3 -> 22.2, 29.4 -> 23.7, 34.1 -> 25.4, 44.5 -> 29.8   524 K rows 86 -> 94, 107 -> 108, 128 -> 112, 202 -> 132; 1 M rows 184 -> 178, 240 -> 199, 287 -> 209, 396 -> 247
//          f16 x 128    24.2 -> 24.2, 29.7 -> 27.1, 34.5 -> 29.5, 44.4 -> 34.3   524 K rows 89 -> 103, 112 -> 117, 133 -> 128, 203 -> 148; 1 M rows 184 -> 193, 241 -> 217, 289 -> 233, 396 -> 278
//   SpMM   f32 x 128    35 -> 34, 43 -> 39, 50 -> 41, 67 -> 46        524 K rows 200 -> 161, 254 -> 186, 293 -> 191, 384 -> 217
//          f32 x 64     19.7 -> 22.1, 23.4 -> 24.1, 27.2 -> 25.1, 35.5 -> 27.9   717 K rows 91 -> 104, 144 -> 139, 203 -> 143, 271 -> 166; 1 M rows 196 -> 175, 253 -> 198, 289 -> 203, 381 -> 231
//          f16 x 128    23.9 -> 27.5, 28.7 -> 31.7, 32.8 -> 33.3, 41 -> 40       717 K rows 116 -> 156, 188 -> 184, 265 -> 195, 338 -> 228; 1 M rows 272 -> 223, 339 -> 261, 383 -> 272, 473 -> 318
//          f64 x 32     22.4 -> 29.1, 26.8 -> 30.9, 31.3 -> 32.0, 40 -> 36.8 (1030 chunks); 704 K rows 112 -> 133, 186 -> 152; 1 M rows 208 -> 190, 269 -> 214, 313 -> 219, 411 -> 249
// The number of nonzeros not said: the caller wants the plan used.
struct WindowGain {
    float base, per_slot;
    float larger;       // above larger_mb MiB of dense operands ...
    size_t larger_mb;
    float largest;      // ... and above largest_mb
    size_t largest_mb;
};
inline float window_gain(const PlanRef& plan, int m2, size_t row_bytes, const WindowGain& of)
{
    const float slots = plan.nonzeros < 31ll * m2 ? (float)plan.nonzeros / (float)m2 : 31.f;
    const size_t mb = 2 * (size_t)m2 * row_bytes >> 20;
    return (of.base + of.per_slot * slots) * (mb >= of.largest_mb ? of.largest : mb >= of.larger_mb ? of.larger : 1.f);
}
// (the time of the standard kernels over that of the window kernels)
inline float windows_pay(const PlanRef& plan, int m2, int round, size_t row_bytes, const WindowGain& full_round)
{
    const int chunks = plan.host_counts[0], rounds = (chunks + round - 1) / round;
    return window_gain(plan, m2, row_bytes, full_round) * (float)chunks / ((float)rounds * (float)round);
}

// Do the ring kernels pay for a call?  A strip costs as much as its chunks and a start (the first window, not copied beside any work)
// worth a chunk and half a chunk per slice; few strips with a chunk more than the others do not count.  gain: time of the standard kernels
// over that of a chunk of s slots a row, measured as for the window kernels on bands of 128 to 256 columns and 66 K to 1 M rows (and set so that
// of 2100 such calls, three matrices in turn, two lose more than 2 % against what is taken of standard and window kernels, 3 and 4), SpMM: us,
// standard -> ring, 9 / 14 / 19 / 27 slots a row (the operands within the last-level cache; beyond it the ring gains up to twice that)
//   f32 x 64    131 K 20.2 -> 18.8, 24.3 -> 20.8, 29.6 -> 23.0, 38.2 -> 27.2; 350 K 48 -> 42, 60 -> 48, 75 -> 55, 95 -> 66; 90 K 14.8 -> 18.5, 17.5 -> 20.6, 21.5 -> 22.6, 27.3 -> 26.1
//   f32 x 128   131 K 37 -> 32, 45 -> 37, 57 -> 41, 73 -> 50; 66 K 20.4 -> 20.5, 24.7 -> 23.1, 29.4 -> 25.4, 38.4 -> 30.4; 90 K 26.7 -> 31.4, 32.4 -> 34.8, 39.0 -> 37.7, 51 -> 44
//   f32 x 32    600 K 44 -> 53, 51 -> 58, 66 -> 64, 87 -> 75; 200 K 17.3 -> 22.6, 20.0 -> 24.5, 24.2 -> 26.2, 31.7 -> 30.5
//   f16 x 128   200 K 36 -> 43, 43 -> 47, 54 -> 52, 69 -> 61; 600 K 104 -> 101, 124 -> 112, 150 -> 126;  f16 x 64  600 K 54 -> 66, 68 -> 75, 82 -> 85, 102 -> 101
//   f64 x 32    131 K 21.3 -> 19.7, 25.5 -> 21.6, 31.7 -> 24.5, 40.2 -> 29.1;  f64 x 16  131 K 20.0 -> 14.8, 23.7 -> 16.6, 37.8 -> 21.5 (27)
// and SDDMM (which takes whole rows only):
//   f32 x 64    131 K 24.8 -> 21.7, 29.9 -> 23.8, 35.9 -> 27.2, 46.3 -> 31.6; 350 K 60 -> 48, 74 -> 53, 93 -> 65, 119 -> 79; 600 K 100 -> 100, 124 -> 107, 179 -> 120
//   f32 x 32    350 K 33 -> 40, 41 -> 43, 54 -> 47, 72 -> 55; 600 K 54 -> 65, 68 -> 80, 87 -> 92, 133 -> 107; 1 M 86 -> 126, 125 -> 137, 175 -> 145, 236 -> 171
//   f16 x 128   131 K 25.0 -> 24.4, 30.4 -> 27.6, 37.3 -> 31.4, 46.9 -> 37.8; 600 K 102 -> 111, 125 -> 122, 179 -> 136;  f16 x 64  350 K 34 -> 43, 42 -> 46, 54 -> 52, 72 -> 62
inline float rings_pay(const PlanRef& plan, int m2, int workgroups, int slices, size_t row_bytes, const WindowGain& chunk)
{
    const int parts = plan.host_counts[0] * slices, rounds = (parts - 16 * slices + workgroups - 1) / workgroups;
    return window_gain(plan, m2, row_bytes, chunk) * (float)parts / (((float)rounds + 1.f + 0.5f * (float)slices) * (float)workgroups);
}

// Which kernels take the chunks with a window, for dense rows that a ring takes in `slices` (0: not) and the window kernels take or not.
inline void choose_windows(PlanRef& plan, int m2, int workgroups, int slices, bool window_takes, size_t row_bytes, const WindowGain& of_rings, const WindowGain& of_windows)
{
    if (plan.dev == nullptr) return;
    if (plan.host_counts == nullptr || plan.nonzeros <= 0 || m2 <= 0) {
        // the number of nonzeros not said: the caller wants the plan used, which rows of 128 bytes never were
        plan.rings = slices > 0;
        if (slices > 0 ? row_bytes == 128 : !window_takes) plan.no_window();
        return;
    }
    const float rings = slices > 0 ? rings_pay(plan, m2, workgroups, slices, row_bytes, of_rings) : 0.f;
    const float windows = window_takes ? windows_pay(plan, m2, workgroups, row_bytes, of_windows) : 0.f;
    // Chunks without a window stay with the standard kernels, which work on the others as well while the dense rows of those are on their way: what
    // is taken from them saves less than its share.  Rings in the place of window kernels are faster all the same (1 M rows x 64, 27 slots, one
    // chunk in ten / two in five without a window, runs of 110 / 73 chunks: standard 421 / 555, windows 359 / 578, rings 321 / 552), but else they are
    // for matrices with nearly no such chunk: up to a twentieth, of rows of 128 bytes, which the window kernels do not take, as many hundredths
    // as they have slots above 21 (x 32, 27 slots, a twentieth, runs of 110 / 14 chunks: 203 -> 177, 195 -> 190; a tenth 218 -> 205, 195 -> 219).
    const long long chunks = plan.host_counts[0], without = chunks - plan.host_counts[1];
    const bool together = without == 0 || (window_takes ? 20 * without <= chunks || windows >= 1.f : 100 * without * m2 <= (plan.nonzeros - 21ll * m2) * chunks);
    // (of both, up to four rounds the better one; beyond it the dense operands come from memory, and the rings copy less: 131 K rows of 16
    // x 128 39 windows, 41 rings; 350 K of 12 halves x 128 90 and 75)
    plan.rings = rings >= 1.f && together && (chunks > 4 * workgroups || rings >= windows);
    if (!plan.rings && windows < 1.f) plan.no_window();
}

hipError_t group_plan_launch(int M, const int* row_ptr, const int* col, int* plan, hipStream_t stream);

// The attention kernels take nheads problems on one pattern of M rows, N columns and nnz
// nonzeros per launch (operands head after head).  (plan: only a group plan is used)
template <typename T>
hipError_t attention_launch(int nheads, int M, int N, int nnz, int d, const int* row_ptr, const int* col, const float* val,
                            const T* q, const T* k, const T* v, float scale, float* out, float* probs, float* row_stats,
                            PlanRef plan, hipStream_t stream);

constexpr bool attention_tiles_fit(int N, size_t row_bytes) { return N > 0 && (size_t)N * row_bytes < (1ull << 32); }
// Do the tiles of a group plan go to the tile kernels?  (They address a head's k and v with 32-bit offsets; N = 0: not said, one head.)
// Where the other kernel is the one for groups (groups_min, the pass's own figure), always: 4500 rows of 200 columns in fp32, width 32 / 64
// / 128: 17 -> 14, 24 -> 18, 70 -> 28 us.  Where it is a wave per row, from 1.5 M nonzeros over all heads on: a tile takes 10 to 45 us
// however few there are, and rows in no tile are a launch more.  Us row by row -> on tiles, fp32 / halves: 4096 rows of 256 and 64 random
// columns, a few rows left over, 1.3 M nonzeros, width 64: 25.4 -> 26.5 / 15.7 -> 19.1, 128: 48.9 -> 47.7 / 25.7 -> 24.9; 3000 of 200 and
// 16, 1.3 M: 28.7 -> 22.0 / 17.6 -> 14.7, 54.4 -> 37.5 / 29.1 -> 19.5, 0.65 M: 16.3 -> 17.6 / 10.7 -> 13.2, 27.1 -> 26.2 / 16.7 -> 15.7.
// Where the tiles have all rows (but for fp32 of width 32: 2048 rows of 600 and 96, 1.4 M, 16.3 -> 17.1):
//   * more than 64 tiles over all heads (with up to 1024 rows every wave of the other kernel has a SIMD of its own), from 0.4 M on: 1280
//     rows of 400 and 64, width 64 19.5 -> 18.2 / 12.7 -> 10.9, 128 34.2 -> 29.5 / 19.8 -> 15.3; 2000 of 250 12.0 -> 10.7 / 8.5 -> 6.9,
//     20.4 -> 15.7 / 12.6 -> 8.6; 2800 of 400 23.4 -> 13.9 / 14.7 -> 7.7, 41.7 -> 20.8 / 24.3 -> 10.0; halves of width 32 from 0.6 M: 2000
//     of 250 and 20 7.0 -> 7.6, 2800 of 250 7.0 -> 6.2;
//   * fewer, with 700 nonzeros a row, from 0.4 M on but not in fp32 of width 64: 1024 rows of 800 and 64, width 64 22.5 -> 25.9 / 17.1 ->
//     13.4, 128 48.4 -> 41.6 / 23.9 -> 19.5, halves of width 32 13.1 -> 11.1; of 400 and 64 14.5 -> 18.2 / 11.6 -> 10.8, 26.1 -> 28.7 /
//     14.5 -> 15.2, 8.5 -> 9.3, training step 68 -> 74 / 64 -> 67.
inline bool attention_uses_tiles(const PlanRef& plan, int groups_min, int nheads, int N, long long nnz, size_t row_bytes, bool halves)
{
    if (plan.groups == nullptr || plan.group_counts == nullptr || plan.group_counts[1] <= 0 || plan.group_counts[3] <= 0) return false;
    const long long tiles = plan.group_counts[3];
    const bool all_rows = plan.group_counts[2] == 0 && 4 * tiles == plan.group_counts[1];
    long long enough = 1500000;
    if (all_rows && (halves || row_bytes > 128)) {
        if (tiles * nheads > 64)
            enough = row_bytes > 64 ? 400000 : 600000;
        else if (nnz >= 700 * 16 * tiles && (halves || row_bytes > 256))
            enough = 400000;
    }
    return (plan.group_counts[1] >= groups_min || nnz * nheads >= enough) && attention_tiles_fit(N, row_bytes);
}
// (rode_attention_tile.hip) the rows of a group plan's tiles, the same arguments; plan: the group plan
template <typename T>
hipError_t attention_tiles_launch(int nheads, int M, int N, int nnz, int d, const int* row_ptr, const int* col, const float* val,
                                  const T* q, const T* k, const T* v, float scale, float* out, float* probs, float* row_stats,
                                  const int* plan, int plan_fours, hipStream_t stream);

// Gradient of the attention kernel (rode_attention_backward.hip): the row pass over the
// pattern, then the column pass over the transposed pattern (plan: only a group plan is used,
// of the pattern the pass walks).  pz: nheads x 2 * nnz floats, written by the first in the
// order of the transposed pattern (t_slot: every nonzero's slot there), read by the second.
// row_stats: NULL when probs holds probabilities, else what attention_launch wrote beside the
// scores in probs.
template <typename T>
hipError_t attention_backward_rows_launch(int nheads, int M, int N, int nnz, int d, const int* row_ptr, const int* col,
                                          const float* val, const float* probs, const float* row_stats, const float* g,
                                          const float* out, const T* k, const T* v, float scale, const int* t_slot, float* dq,
                                          float* pz, PlanRef plan, hipStream_t stream);
// (rode_attention_backward_tile.hip) the row pass for the rows of a group plan's tiles; plan: the group plan
template <typename T>
hipError_t attention_backward_tiles_launch(int nheads, int M, int N, int nnz, int d, const int* row_ptr, const int* col, const float* val,
                                           const float* probs, const float* row_stats, const float* g, const float* out, const T* k,
                                           const T* v, float scale, const int* t_slot, float* dq, float* pz, const int* plan,
                                           hipStream_t stream);

// (rode_attention_backward_cols_tile.hip) the column pass for the tiles of a group plan of the transposed pattern; plan: that plan
template <typename T>
hipError_t attention_backward_cols_tiles_launch(int nheads, int M, int N, int nnz, int d, const int* t_row_ptr, const int* t_col,
                                                const float* pz, const float* g, const T* q, float* dk, float* dv, const int* plan,
                                                hipStream_t stream);

template <typename T>
hipError_t attention_backward_cols_launch(int nheads, int M, int N, int nnz, int d, const int* t_row_ptr, const int* t_col,
                                          const float* pz, const float* g, const T* q, float* dk, float* dv, PlanRef plan,
                                          hipStream_t stream);

hipError_t hub_plan_launch(int M, int dense_rows, int nnz, int min_len, const int* row_ptr, int* plan, hipStream_t stream);
hipError_t hub_pieces_launch(int hub_rows, int dense_rows, const int* row_ptr, const int* col, int* plan, hipStream_t stream);

size_t window_plan_ints(int m2);
size_t window_plan_rows_bytes(int m2);
// (header_counts: null, or where the last workgroup writes the header's four ints; the header itself is then cleared already,
// by preprocess_launch, which has `chunks` from window_plan_chunks)
int window_plan_chunks(int m2);
hipError_t window_plan_header_launch(int m2, int windowed, int* plan, hipStream_t stream);
hipError_t window_plan_launch(int m2, int dense_rows, const int* residue_rows, const int* row_ptr, const int* col,
                              int* plan, hipStream_t stream, int* header_counts = nullptr);
hipError_t window_plan_rows_launch(int m2, const int* residue_rows, const int* row_ptr, const int* col, const int* plan,
                                   void* rows, hipStream_t stream);

// (rode_spmm.hip) which rows an SpMM call under kSpmmOverwrite stores instead of adding to
int spmm_overwrite_limit(int m1, bool hub_plan);
size_t spmm_hub_partial_rows(const int* hub_counts, int n, int acc_bytes);
template <typename T>
hipError_t spmm_launch(int m1, int m2, int n, const int* block_rows, const int* residue_rows, const int* st_off,
                       const int* row_ptr, const int* col, const typename SpmmAcc<T>::type* val, const T* B,
                       typename SpmmAcc<T>::type* C, int flags, PlanRef plan, hipStream_t s1, hipStream_t s2);

// the window kernel of SpMM over the planned chunks of the residue list
template <typename T>
hipError_t spmm_window_launch(int m2, int n, int owned_slots, const int* col, const typename SpmmAcc<T>::type* val, const T* B,
                              typename SpmmAcc<T>::type* C, const PlanRef& plan, hipStream_t stream);

// (stored: rows of at most that many aligned slots are left alone as well)
hipError_t spmm_clear_rows_launch(int M, size_t row_bytes, int stored, const int* row_ptr, void* C, hipStream_t stream);

template <typename T>
hipError_t sddmm_launch(int m1, int m2, int k, const int* block_rows, const int* residue_rows, const int* st_off,
                        const int* row_ptr, const int* col, const float* val, const T* lhs, const T* rhs,
                        float* out, PlanRef plan, hipStream_t s1, hipStream_t s2);

// the window kernel of SDDMM over the planned chunks of the residue list
template <typename T>
hipError_t sddmm_window_launch(int m2, int k, const int* col, const float* val, const T* lhs, const T* rhs, float* out,
                               const PlanRef& plan, hipStream_t stream);

hipError_t permute_launch(int n, const float* src, const int* index, float* dst, hipStream_t stream);
size_t csr_transpose_workspace_bytes(int nnz);
hipError_t csr_transpose_launch(int M, int N, int nnz, const int* row_ptr, const int* col, int* t_row_ptr, int* t_col,
                                int* perm, void* workspace, hipStream_t stream);
hipError_t csr_softmax_launch(int M, const int* row_ptr, const float* in, float* out, float scale,
                              hipStream_t stream);
hipError_t csr_softmax_backward_launch(int M, const int* row_ptr, const float* p, const float* dp, float* ds,
                                       float scale, hipStream_t stream);

} // namespace rode
