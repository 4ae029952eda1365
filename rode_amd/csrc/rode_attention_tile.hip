// Sparse attention, forward, for the tiles of 16 rows of a group plan (sliding windows and
// other masks whose adjacent rows share long runs of consecutive columns), on the matrix cores:
//     out[r, :] = sum_idx p[idx] * v[col(idx), :],   p = softmax of scale * values[idx] * <q[r, :], k[col(idx), :]>
// (the contract of rode_attention.hip, whose kernels take the rows of no tile).
//
// One workgroup per tile and head.  Its four waves take the columns of the run 16 or 32 at a time, in
// turn (score products of 16 x 16, a running softmax, D / 16 weighted-sum products; layouts in
// rode_tile.hpp), and then the nonzeros outside the run of four rows each, side by side, 64 of every row at a time
// (TileOutside); every wave, and every row outside its run, has a softmax of its own,
// and the partial results meet in LDS.  Columns at the ends of the range that a row does not hold get
// probability zero.  A non-finite row of v there would reach rows that do not reference it
// (0 * Inf), and shows as a non-finite result: the tile's rows are then computed again, all of them
// row by row.
//
// Measured (16 384 rows, window 512 and 64 random columns, width 64): eight heads of halves 0.552 ms with four rows at a time on
// the vector ALUs, 0.206 here, 0.176 with four tiles a workgroup, which take that call now (attention_wide_kernel); eight heads in fp32 0.693 -> 0.39.
// No rate was at its limit with those halves: the vector ALUs issued 66 % of the time (a fifth of it the tiles' prologues, once per
// head), the address units were busy for 63 %, 3.2 GB left the L2s and 0.62 GB passed them (3.1 TB/s); 2.7 waves per SIMD waited for memory
// 48 % of their time (all before LDS transposed on the way out).  What was slow on
// the way: dense rows and values loaded straight into operand layout (adjacent lanes on different rows: 64 clocks of the
// memory pipe per load, 0.38 ms); the nonzeros outside the run of one row after the other (us, fp32 / halves of width 64, one head:
// 75 / 36 -> 69 / 34, width 128 164 / 68 -> 131 / 58; 20 000 rows of 300 and 96 random columns 121 / 62 -> 97 / 55, width 128 274 / 129 ->
// 196 / 100; eight heads of halves 222 -> 209).  (The extent of a row outside its run waits in LDS: in registers it
// cost halves of width 64 a wave per SIMD, 248 us.)
//
// 32-bit operands use the 32-bit matrix instructions (exact products, 157 TFLOP/s against 79 on the
// vector ALUs); 16-bit operands split the probabilities into two halves each (TileWeights).  Errors against 64 bits of
// the output and of the gradients that follow from it, against those of the kernels on the vector ALUs (2-norms, masks of
// 200 to 700 columns, widths 32 to 128, scores with a deviation of 1 and of 8): fp32 0.72 to 1.03 times, halves 0.82 to
// 1.01 times.  That took sums in trees (mma_rows, TileCols), exponents that are rounded once (TileSoftmax) and row
// sums of the 32-bit weights on the vector ALUs; as chains of matrix products with a rounded offset in the exponent it
// was 1.4 to 3.1 and 1.0 to 1.7 times.
#include "rode_tile.hpp"
#include "rode_units.hpp"
#include "rode_internal.hpp"

#include <type_traits>

namespace rode {

namespace {

// With 32-bit operands, when a head's k and v are of that size and more (an L2 has 4 MB), the nonzeros outside the runs come before
// the columns of the runs: the workgroups then begin with them together, all of them at rows of k, then all at rows of v, and find
// more of those in L2.  us, after the runs -> before them: 16 384 rows, window 512 and 64 random columns, width 64 66.6 -> 60.1, four heads 225 -> 202, 128 129
// -> 123; 20 000 of 128 and 16, four heads 112 -> 98; 14 000 of 400 and 32 (7.2 MB) 47.4 -> 45.2; 12 000 (6.1 MB) 33.2 -> 36.3, four
// heads 112 -> 111; 9000 (4.6 MB) 35.5 -> 38.0; width 32, 16 384 rows (4.2 MB) 31.1 -> 34.0.  (Halves: no faster at any size; the gradient's
// two passes: row pass 97 either way, column pass 73, with halves 1 to 3 % slower.)
constexpr size_t kOutsideFirstBytes = 7000000;

// Running softmax of the rows of a tile: 4 or 8 scores of this lane's row at a time (-inf: none).  A weight is exp(score)
// over a power of two, 2^ref, the first one that no score so far passes: the exponent of a weight is then a single rounding away
// from score * log2(e), and the steps and the waves rescale each other's sums exactly.  PARTS: the sums of a few steps are put away
// into `total` (a wave with all columns of a run: one chain of 6 / 18 steps had 1.13 / 1.36 times the error of four chains put
// together, parts of four steps up to 1.05, those of attention_wide_kernel 0.95 to 1.00; 16 heads of 2048 and 4096 rows, halves).
template <typename T, int D, bool PARTS = false>
struct TileSoftmax {
    static constexpr int N = 4 * tile_blocks<T>();
    float m = -INFINITY;      // largest score of the row (the same in its four lanes)
    float ref = -0x1p126f;    // (no score yet)
    float l = 0.f;            // sum of this lane's weights
    f32x4 acc[D / 16];        // weighted sums, times TileWeights<T>::kScale
    float total_ref = -0x1p126f, total_l = 0.f;
    f32x4 total[PARTS ? D / 16 : 1];
    __device__ __forceinline__ TileSoftmax()
    {
#pragma unroll
        for (int b = 0; b < D / 16; ++b) acc[b] = kNothing;
#pragma unroll
        for (int b = 0; PARTS && b < D / 16; ++b) total[b] = kNothing;
    }
    __device__ __forceinline__ void put_away()
    {
        const float corr = __builtin_amdgcn_exp2f(total_ref - ref);
        total_ref = ref;
#pragma unroll
        for (int b = 0; b < D / 16; ++b) {
#pragma unroll
            for (int i = 0; i < 4; ++i) total[b][i] = fmaf(total[b][i], corr, acc[b][i]); // (corr: a power of two)
            acc[b] = kNothing;
        }
        total_l = fmaf(total_l, corr, l);
        l = 0.f;
    }
    __device__ __forceinline__ void step(const float (&sc)[N], TileWeights<T>& weights)
    {
        float top = sc[0];
#pragma unroll
        for (int j = 1; j < N; ++j) top = fmaxf(top, sc[j]);
        m = fmaxf(m, quad_max(top));
        const float now = m == -INFINITY ? ref : ceilf(m * kLog2e);
        if (__any(now != ref)) {
            const float corr = __builtin_amdgcn_exp2f(ref - now);
            l *= corr;
#pragma unroll
            for (int b = 0; b < D / 16; ++b) acc[b] *= corr;
            ref = now;
        }
        float p[N], sum[N];
#pragma unroll
        for (int j = 0; j < N; ++j) sum[j] = p[j] = __builtin_amdgcn_exp2f(fmaf(sc[j], kLog2e, -ref));
#pragma unroll
        for (int h = N / 2; h >= 1; h /= 2)
#pragma unroll
            for (int j = 0; j < h; ++j) sum[j] += sum[j + h];
        l += sum[0];
        weights.set(p, TileWeights<T>::kScale); // (the scale not in the exponent, which would lose digits to it)
    }
    // (a score beyond the range of the powers of two gives none of its row a weight)
    __device__ __forceinline__ bool finite() const { return all_finite<D / 16>(acc) && (!PARTS || all_finite(total)) && fabsf(ref) <= 0x1p126f; }
};

// Four rows of a tile (the quarter'th four; the tile's first row: row0) without the nonzeros of their runs (or, `whole`, with them),
// 64 of each row at a time: 16 lanes have a row's nonzeros, LPR lanes read a dense row, 16 bytes each, every lane group the
// rows of its own LPR nonzeros.  The scores of all 64 first, then their rows of v.  staging: 2 * kOutsideSteps * kWave floats of
// the wave's own; the four weighted sums go to `to`, D + 4 floats apart, maximum and sum of weights of row r of the tile to to_m[r] and to_l[r].
template <typename T, int D, int KEEP>
__device__ __forceinline__ void rows_outside(const int4* extents, int quarter, int row0, bool whole, int lane, const int* __restrict__ col,
                                             const float* __restrict__ val, const T* __restrict__ q, const T* __restrict__ k,
                                             const T* __restrict__ v, float scale, float* probs, float* staging, float* to, float* to_m, float* to_l)
{
    using Out = TileOutside<T, D>;
    constexpr int VEC = Out::kVec, LPR = Out::kLpr, RPG = Out::kRows, QUADS = Out::kQuads, S = kOutsideSteps;
    const int ls = lane % LPR, group = lane / LPR;
    const unsigned lane_at = ls * 16u; // (an operand of a tile is at most 4 GB: 32-bit offsets)
    const char* k_bytes = reinterpret_cast<const char*>(k);
    const char* v_bytes = reinterpret_cast<const char*>(v);
    unsigned* my_at = reinterpret_cast<unsigned*>(staging);
    float* my_p = staging + S * kWave;
    const Out of(extents, quarter, lane, whole);
    typename DotVec<T>::Reg a[RPG][1][DotVec<T>::kRegs];
#pragma unroll
    for (int i = 0; i < RPG; ++i) load_lhs_slice<T, D, 1, false>(q, row0 + of.row(i), D, lane, a[i]);
    float m_run = -INFINITY, l_lane = 0.f, acc[RPG][VEC];
#pragma unroll
    for (int i = 0; i < RPG; ++i)
#pragma unroll
        for (int x = 0; x < VEC; ++x) acc[i][x] = 0.f;
#pragma unroll 1
    for (int off = 0; off < of.most; off += 16 * S) {
        float w[S], sc[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            int c = 0;
            w[s] = 0.f;
            if (off + 16 * s < of.cnt) { // (lanes past the end repeat the last nonzero with probability 0)
                const int idx = of.slot(off + 16 * s + lane % 16);
                c = col[idx];
                w[s] = val[idx];
            }
            my_at[s * kWave + lane] = (unsigned)c * (unsigned)(D * sizeof(T));
        }
        wave_lds_sync();
#pragma unroll
        for (int s = 0; s < S; ++s) {
            float d = 0.f;
#pragma unroll
            for (int i = 0; i < RPG; ++i)
                if (off + 16 * s < of.cnt_of[i]) {
                    uint4 k_part[QUADS][4];
#pragma unroll
                    for (int u = 0; u < QUADS; ++u) {
                        const u32x4 o = *reinterpret_cast<const u32x4*>(my_at + s * kWave + group * LPR + 4 * (i * QUADS + u));
#pragma unroll
                        for (int j = 0; j < 4; ++j) k_part[u][j] = *reinterpret_cast<const uint4*>(k_bytes + (o[j] + lane_at));
                    }
#pragma unroll
                    for (int u = 0; u < QUADS; ++u) {
                        float p[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) p[j] = DotVec<T>::dot_raw(a[i][0], k_part[u][j], 0.f);
                        const float sum = sddmm_quad_reduce<LPR>(p, ls);
                        if ((ls >> 2) == i * QUADS + u) d = sum;
                    }
                }
            const int slot = off + 16 * s + lane % 16;
            sc[s] = slot < of.cnt ? scale * (w[s] * d) : -INFINITY;
            if (KEEP != kKeepNothing && slot < of.cnt) probs[of.slot(slot)] = sc[s];
        }
        // the running softmax of the row (the same in its 16 lanes but for l_lane)
        float top = sc[0];
#pragma unroll
        for (int s = 1; s < S; ++s) top = fmaxf(top, sc[s]);
        const float m_new = fmaxf(m_run, butterfly_max<1, 16>(top));
        const float m_safe = m_new == -INFINITY ? 0.f : m_new;
        const float corr = __expf(m_run - m_safe);
        m_run = m_new;
        float p_sum = 0.f;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const float p = off + 16 * s + lane % 16 < of.cnt ? __expf(sc[s] - m_safe) : 0.f;
            p_sum += p;
            my_p[s * kWave + lane] = p;
        }
        l_lane = fmaf(l_lane, corr, p_sum);
        if (off > 0) { // (nothing to rescale before)
            const float corr_of[2] = {RPG > 1 ? lane_pair16(corr).a : corr, RPG > 1 ? lane_pair16(corr).b : corr};
#pragma unroll
            for (int i = 0; i < RPG; ++i)
#pragma unroll
                for (int x = 0; x < VEC; ++x) acc[i][x] *= corr_of[i];
        }
        wave_lds_sync();
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < RPG; ++i)
                if (off + 16 * s < of.cnt_of[i]) Out::add(v_bytes, lane_at, my_at + s * kWave, my_p + s * kWave, group * LPR + 4 * i * QUADS, acc[i]);
        wave_lds_sync();
    }
    const float l = butterfly_sum<1, 16>(l_lane);
    of.store(acc, to, D + 4, lane);
    if (lane % 16 == 0) to_m[of.mine] = m_run, to_l[of.mine] = l;
}

// A step's kStep columns from c0 on for a tile's 16 rows: the staged rows of k and v and values (in the order of the scores: lds_w),
// `in`: every row of the tile holds every one of the columns.  f_a, f_end, f_base: the run of the row that this lane has in memory's order.
template <typename T, int D, int KEEP, bool PARTS>
__device__ __forceinline__ void columns_step(const u32x4* lds_k, const u32x4* lds_v, f32x4* lds_w, int c0, bool in, int lane, const TileLane& me,
                                             int f_a, int f_end, int f_base, const TileRow<T, D>& q_row, float scale, float* probs, TileSoftmax<T, D, PARTS>& sm)
{
    constexpr int NT = tile_blocks<T>();
    using KStage = TileStage<T, D, kAlong>;
    using VStage = TileStage<T, D, tile_columns<T>()>;
    const int gq = lane / 16;
    float sc[4 * NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        TileRow<T, D> k_row;
        KStage::read(lds_k, t, lane, k_row);
        const f32x4 dot = mma_rows<T, D>(k_row, q_row), w = TileSquare<T>::as_scores(lds_w, t, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[4 * t + i] = scale * (w[i] * dot[i]);
    }
    if (KEEP != kKeepNothing) { // the scores leave in the order of the values
#pragma unroll
        for (int t = 0; t < NT; ++t) TileSquare<T>::as_scores(lds_w, t, lane) = f32x4{sc[4 * t], sc[4 * t + 1], sc[4 * t + 2], sc[4 * t + 3]};
        wave_lds_sync();
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const f32x4 out4 = TileSquare<T>::in_order(lds_w, t, lane);
            const int c = c0 + 16 * t + lane % 4 * 4;
            if (in) {
                *reinterpret_cast<f32x4_u*>(probs + f_base + c) = out4;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (c + i >= f_a && c + i < f_end) probs[f_base + c + i] = out4[i];
            }
        }
    }
    if (!in) {
#pragma unroll
        for (int j = 0; j < 4 * NT; ++j) {
            const int c = c0 + 16 * (j / 4) + 4 * gq + j % 4;
            sc[j] = c >= me.a && c < me.a + me.len ? sc[j] : -INFINITY;
        }
    }
    TileWeights<T> weights;
    sm.step(sc, weights);
    TileCols<T, D> v_cols;
    v_cols.load(lds_v, lane);
    v_cols.accumulate(weights, sm.acc);
}

template <typename T, int D, int KEEP>
__global__ void __launch_bounds__(kWgThreads, (D == 128 ? 2 : tile_waves<T, D>()))
attention_tile_kernel(int n_tiles, const RowTile* __restrict__ tiles, const int* __restrict__ runs,
                      const int* __restrict__ row_ptr, const int* __restrict__ col, const float* __restrict__ val,
                      const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, float scale,
                      float* __restrict__ out, float* probs, float2* __restrict__ stats, bool outside_first, HeadStrides heads)
{
    constexpr int NB = D / 16, PAD = D + 4, NT = tile_blocks<T>(), kStep = 16 * NT;
    using KStage = TileStage<T, D, kAlong>;
    using VStage = TileStage<T, D, tile_columns<T>()>;
    // Per wave: staged rows of k and v and the values of a step.  Once the columns of the run are done: staging for the nonzeros
    // outside, then the wave's partial result and behind it the results of its four rows outside their runs.
    constexpr int kPart = kTileRows * PAD, kStageFloats = 2 * KStage::kBytes / 4 + TileSquare<T>::kFloats;
    static_assert(kPart + kOutsideRows * PAD <= kStageFloats && 2 * kOutsideSteps * kWave <= kStageFloats, "what comes later fits");
    __shared__ __attribute__((aligned(16))) float shared[kWavesPerWg][kStageFloats];
    __shared__ float part_m[kWavesPerWg + 1][kTileRows], part_l[kWavesPerWg + 1][kTileRows]; // (the last: outside the runs)
    __shared__ float part_ref[kWavesPerWg][kTileRows];
    constexpr bool kMayBeFirst = sizeof(T) == 4; // (outside_first)
    __shared__ __attribute__((aligned(16))) float ahead[kMayBeFirst ? kWavesPerWg * kOutsideRows * PAD : 4];
    __shared__ int4 extents[kTileRows]; // (for the nonzeros outside the runs: not in registers until then)
    const int tile = xcd_logical_block(blockIdx.x, gridDim.x);
    if (tile >= n_tiles) return;
    const RowTile rt = tiles[tile];
    if (rt.hi <= rt.lo) return; // not a tile: other kernels have its rows
    q = of_head(q, heads.rows), k = of_head(k, heads.cols), v = of_head(v, heads.cols);
    out = of_head(out, heads.rows), probs = of_head(probs, heads.nnz), stats = of_head(stats, heads.rows / D);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave; // (uniform: scalar registers)
    const int n = lane % 16, gq = lane / 16;
    const TileLane me = tile_lane(tile * kTileRows + n, row_ptr, runs);
    const int base = me.base();
    if (threadIdx.x < kTileRows) extents[threadIdx.x] = me.packed();
    // the sums of the nonzeros outside the runs: behind the wave's own in the steps' staging, or, where they may come first, apart
    float* outside = kMayBeFirst ? ahead + wave * kOutsideRows * PAD : shared[wave] + kPart;
    auto rows_outside_runs = [&](bool whole) __attribute__((always_inline)) {
        int here = lane; // (nothing worked out from it before is worth a register until then)
        asm volatile("" : "+v"(here));
        rows_outside<T, D, KEEP>(extents, wave, tile * kTileRows, whole, here, col, val, q, k, v, scale, probs, shared[wave], outside,
                                 part_m[kWavesPerWg], part_l[kWavesPerWg]);
    };
    if (kMayBeFirst && outside_first) {
        __syncthreads(); // (extents)
        rows_outside_runs(false);
    }
    const int steps = (rt.hi - rt.lo + kStep - 1) / kStep;
    u32x4* lds_k = reinterpret_cast<u32x4*>(shared[wave]);
    u32x4* lds_v = lds_k + KStage::kBytes / 16;
    f32x4* lds_w = reinterpret_cast<f32x4*>(lds_v + VStage::kBytes / 16);
    TileRow<T, D> q_row;
    q_row.load(q + (size_t)me.row * D, gq);
    TileSoftmax<T, D> sm;

    // a step's columns of the run, on their way
    KStage k_rows;
    VStage v_rows;
    f32x4 w_rows[NT];
    // (the row and the four columns that this lane fetches values of: TileSquare)
    const int f_a = __shfl(me.a, lane / 4, kWave), f_end = f_a + __shfl(me.len, lane / 4, kWave), f_base = __shfl(base, lane / 4, kWave);
    auto inside = [&](int c0) { return c0 >= rt.core_lo && c0 + kStep <= rt.core_hi; }; // does every row hold every one of them?
    auto fetch = [&](int c0) __attribute__((always_inline)) {
        const bool in = inside(c0);
        k_rows.load(k + (size_t)c0 * D, rt.hi - 1 - c0, in, lane); // (columns past the range repeat its last)
        v_rows.load(v + (size_t)c0 * D, rt.hi - 1 - c0, in, lane);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int c = c0 + 16 * t + lane % 4 * 4;
            if (in) {
                w_rows[t] = *reinterpret_cast<const f32x4_u*>(val + f_base + c);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) w_rows[t][i] = c + i >= f_a && c + i < f_end ? val[f_base + c + i] : 0.f;
            }
        }
    };
    auto run_columns = [&]() __attribute__((always_inline)) {
        if (wave < steps) fetch(rt.lo + wave * kStep);
        for (int it = wave; it < steps; it += kWavesPerWg) {
            const int c0 = rt.lo + it * kStep;
            const bool in = inside(c0);
            k_rows.store(lds_k, lane);
            v_rows.store(lds_v, lane);
#pragma unroll
            for (int t = 0; t < NT; ++t) TileSquare<T>::in_order(lds_w, t, lane) = w_rows[t];
            wave_lds_sync();
            if (it + kWavesPerWg < steps) fetch(c0 + kWavesPerWg * kStep); // (in flight during this step)
            columns_step<T, D, KEEP, false>(lds_k, lds_v, lds_w, c0, in, lane, me, f_a, f_end, f_base, q_row, scale, probs, sm);
            wave_lds_sync();
        }
    };

    run_columns();
    const bool again = __syncthreads_or(!sm.finite());
    if (again) sm = TileSoftmax<T, D>();
    if (!(kMayBeFirst && outside_first) || again) rows_outside_runs(again); // (the steps' staging is free)

    // the partial results, a wave's relative to its power of two, those outside the runs to the exponential of their maximum
    float* part = shared[wave];
    const float l_row = quad_sum(sm.l);
    if (gq == 0) part_m[wave][n] = sm.m, part_ref[wave][n] = sm.ref, part_l[wave][n] = l_row;
#pragma unroll
    for (int c = 0; c < NB; ++c) *reinterpret_cast<f32x4*>(part + n * PAD + TileCols<T, D>::at(c, gq)) = TileCols<T, D>::sums(sm.acc, c);
    __syncthreads();
    const int r = threadIdx.x / 16, e0 = threadIdx.x % 16 * NB, row = tile * kTileRows + r;
    float top = part_m[0][r];
#pragma unroll
    for (int w = 1; w <= kWavesPerWg; ++w) top = fmaxf(top, part_m[w][r]);
    const float top_safe = top == -INFINITY ? 0.f : top;
    const float* outside_of_row = (kMayBeFirst ? ahead + r / kOutsideRows * kOutsideRows * PAD : shared[r / kOutsideRows] + kPart) + r % kOutsideRows * PAD;
    float f = __builtin_amdgcn_exp2f((part_m[kWavesPerWg][r] - top_safe) * kLog2e);
    float total = part_l[kWavesPerWg][r] * f, o[NB];
#pragma unroll
    for (int x = 0; x < NB; ++x) o[x] = outside_of_row[e0 + x] * f;
#pragma unroll
    for (int w = 0; w < kWavesPerWg; ++w) {
        f = __builtin_amdgcn_exp2f(-fmaf(top_safe, kLog2e, -part_ref[w][r]));
        total = fmaf(part_l[w][r], f, total);
        f *= 1.f / TileWeights<T>::kScale;
#pragma unroll
        for (int x = 0; x < NB; ++x) o[x] = fmaf(shared[w][r * PAD + e0 + x], f, o[x]);
    }
    const float inv = 1.0f / total;
#pragma unroll
    for (int x = 0; x < NB; x += 2)
        *reinterpret_cast<float2*>(out + (size_t)row * D + e0 + x) = make_float2(o[x] * inv, o[x + 1] * inv);
    if (KEEP == kKeepScores && threadIdx.x % 16 == 0) stats[row] = make_float2(top_safe, inv);
    if (KEEP == kKeepProbs) {
        // what the waves wrote are scores: normalised in place
        __threadfence_block();
        __syncthreads();
        const int s = row_ptr[row], e = row_ptr[row + 1];
        for (int slot = s + threadIdx.x % 16; slot < e; slot += 16) probs[slot] = __expf(probs[slot] - top_safe) * inv;
    }
}

// Four neighbouring tiles (64 rows) whose runs lie together, a wave for each: a step's rows of k and v are staged once for the
// four, nothing is put together across waves, and what a tile does once it does in one wave instead of four.  Workgroup after
// workgroup of one head, on one XCD at a time where there are as many heads: its L2 then has one head's k and v.
// The workgroups take their steps so that those of an XCD are at the same columns at the same time (a run's columns in turn, beginning
// with a multiple of their number): a row of k or v then comes out of memory once an XCD and not once in every few of the 9
// workgroups that want it.
//
// Measured (halves, 16 384 rows, eight heads of width 64): window 512 106 -> 76 us (2.9 M lines past the L2s, 370 MB, four fifths of it
// values, which every head reads for itself), and 64 random columns 207 -> 176 (6.95 M lines read and 34 MB written past the L2s, 922 MB: 5.2 TB/s of
// the 6.5 to 7 that pass them; 72 % of the requests hit).  The lines are not all of it: where k and v are one array 3.9 M are read, 533 MB,
// and the call takes an eighth less (in one program 165 -> 145).  A build without the products and the softmax took as
// long along the runs; the steps in the order of the columns 83 and 179; as many heads on an XCD as there are 230.
// Tried for the nonzeros outside the runs (us, of 176): the scores of all rows before the rows of v (fewer lines past the L2s, 690 MB, but a wave
// per SIMD less) 176; half of the rows at a time 176; those of every other workgroup before its run 178; all loads of four rows at once 194.
// Values of two steps together 180; values with non-temporal loads 240.
template <typename T, int D, int KEEP>
__global__ void __launch_bounds__(kWgThreads, (D <= 64 ? 4 : 1))
attention_wide_kernel(int nheads, int n_tiles, const RowTile* __restrict__ tiles, const int* __restrict__ runs,
                      const int* __restrict__ row_ptr, const int* __restrict__ col, const float* __restrict__ val,
                      const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, float scale,
                      float* __restrict__ out, float* probs, float2* __restrict__ stats, HeadStrides heads)
{
    constexpr int PAD = D + 4, NT = tile_blocks<T>(), kStep = 16 * NT, NB = D / 16;
    using KStage = TileStage<T, D, kAlong>;
    using VStage = TileStage<T, D, tile_columns<T>()>;
    constexpr int kPieces = KStage::kLoads / 2; // a wave's share of a step's rows: waves 0 and 1 have those of k, 2 and 3 those of v
    static_assert(KStage::kLoads % 2 == 0 && kWavesPerWg == 4, "two waves have a step's rows of k");
    constexpr int kBuffer = 2 * KStage::kBytes / 4, kSquare = TileSquare<T>::kFloats;
    constexpr int kOut = kTileRows * PAD, kStaging = 2 * kOutsideSteps * kWave; // after the runs, per wave
    constexpr int kFloats = 2 * kBuffer + kWavesPerWg * kSquare > kWavesPerWg * (kOut + kStaging) ? 2 * kBuffer + kWavesPerWg * kSquare : kWavesPerWg * (kOut + kStaging);
    __shared__ __attribute__((aligned(16))) float shared[kFloats];
    __shared__ float out_m[kWavesPerWg][kTileRows], out_l[kWavesPerWg][kTileRows];
    __shared__ int4 extents[kWavesPerWg][kTileRows];
    const int quads = (n_tiles + kWavesPerWg - 1) / kWavesPerWg;
    const int item = xcd_logical_block(blockIdx.x, gridDim.x), head = item / quads, quad = item % quads;
    if (head >= nheads) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave; // (uniform: scalar registers)
    RowTile rt{0, 0, 0, 0};
    int lo = 0x7fffffff, hi = 0;
#pragma unroll
    for (int i = 0; i < kWavesPerWg; ++i) {
        const int tile = quad * kWavesPerWg + i;
        if (tile < n_tiles) {
            const RowTile t = tiles[tile];
            if (t.hi > t.lo) lo = min(lo, t.lo), hi = max(hi, t.hi);
            if (i == wave) rt = t;
        }
    }
    if (hi <= lo) return; // no tiles: other kernels have their rows
    const bool mine = rt.hi > rt.lo;
    q += head * heads.rows, k += head * heads.cols, v += head * heads.cols, out += head * heads.rows;
    if (KEEP != kKeepNothing) probs += head * heads.nnz, stats += head * (heads.rows / D);
    const int row0 = (quad * kWavesPerWg + wave) * kTileRows;
    // the columns of the runs, a step's rows staged by all waves together
    TileSoftmax<T, D, true> sm;
    {
        TileLane me{};
        TileRow<T, D> q_row{};
        if (mine) {
            me = tile_lane(row0 + lane % 16, row_ptr, runs);
            q_row.load(q + (size_t)me.row * D, lane / 16);
            if (lane < kTileRows) extents[wave][lane] = me.packed();
        }
        f32x4* lds_w = reinterpret_cast<f32x4*>(shared + 2 * kBuffer + wave * kSquare);
        // a step's rows (this wave's share of them) and values, on their way
        u32x4 rows[kPieces];
        f32x4 w_rows[NT];
        const int f_a = __shfl(me.a, lane / 4, kWave), f_end = f_a + __shfl(me.len, lane / 4, kWave), f_base = __shfl(me.base(), lane / 4, kWave);
        const T* dense = wave < 2 ? k : v;
        const int piece0 = (wave & 1) * kPieces * kWave + lane; // this lane's first 16 bytes of them
        auto inside = [&](int c0) { return c0 >= rt.core_lo && c0 + kStep <= rt.core_hi; };
        auto wanted = [&](int c0) { return c0 < rt.hi && c0 + kStep > rt.lo; };
        auto fetch = [&](int c0) __attribute__((always_inline)) {
            const u32x4* from = reinterpret_cast<const u32x4*>(dense + (size_t)c0 * D);
            const int last = hi - 1 - c0; // (columns past the range repeat its last)
#pragma unroll
            for (int i = 0; i < kPieces; ++i) {
                const int at = piece0 + i * kWave;
                rows[i] = from[min(at / KStage::kPerRow, last) * KStage::kPerRow + at % KStage::kPerRow];
            }
            if (wanted(c0)) {
                const bool in = inside(c0);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int c = c0 + 16 * t + lane % 4 * 4;
                    if (in) {
                        w_rows[t] = *reinterpret_cast<const f32x4_u*>(val + f_base + c);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) w_rows[t][i] = c + i >= f_a && c + i < f_end ? val[f_base + c + i] : 0.f;
                    }
                }
            }
        };
        const int steps = (hi - lo + kStep - 1) / kStep;
        int c_next = lo + (steps - lo / kStep % steps) % steps * kStep;
        fetch(c_next);
        const int part_steps = 1 + steps / 9; // (a step adds to its part twice, a part to the total once: shorter parts than their number)
        int buffer = 0, left = part_steps;
#pragma unroll 1
        for (int it = 0; it < steps; ++it, buffer ^= 1) {
            const int c0 = c_next;
            u32x4* lds_k = reinterpret_cast<u32x4*>(shared + buffer * kBuffer);
            u32x4* lds_v = lds_k + KStage::kBytes / 16;
            const bool now = wanted(c0);
#pragma unroll
            for (int i = 0; i < kPieces; ++i) {
                const int at = piece0 + i * kWave, r = at / KStage::kPerRow, c = at % KStage::kPerRow;
                (wave < 2 ? lds_k : lds_v)[wave < 2 ? KStage::place(r, c) : VStage::place(r, c)] = rows[i];
            }
            if (now) {
#pragma unroll
                for (int t = 0; t < NT; ++t) TileSquare<T>::in_order(lds_w, t, lane) = w_rows[t];
            }
            __syncthreads(); // (a buffer is written again two steps later: all have read it when they come to the barrier in between)
            c_next = c0 + kStep < hi ? c0 + kStep : lo;
            if (it + 1 < steps) fetch(c_next); // (in flight during this step)
            if (now) columns_step<T, D, KEEP, true>(lds_k, lds_v, lds_w, c0, inside(c0), lane, me, f_a, f_end, f_base, q_row, scale, probs, sm);
            if (--left == 0) sm.put_away(), left = part_steps;
        }
        sm.put_away(); // (not left for the end: with the nonzeros outside the runs in between its registers make the kernel a fifth slower)
    }
    __syncthreads();
    if (!mine) return;
    const bool again = __any(!sm.finite());
    if (again) sm = TileSoftmax<T, D, true>();
    const int n = lane % 16, gq = lane / 16;
    float* part = shared + wave * (kOut + kStaging);
#pragma unroll 1
    for (int quarter = 0; quarter < kTileRows / kOutsideRows; ++quarter)
        rows_outside<T, D, KEEP>(extents[wave], quarter, row0, again, lane, col, val, q, k, v, scale, probs, part + kOut, part + quarter * kOutsideRows * PAD,
                                 out_m[wave], out_l[wave]);
    // the two partial results, the run's relative to its power of two, the other to the exponential of its maximum: put together relative
    // to the former where the row's largest score is the run's (its sums, of four waves' before, are not rounded once more for it)
    wave_lds_sync();
    const float m_out = out_m[wave][n], top = fmaxf(sm.m, m_out), top_safe = top == -INFINITY ? 0.f : top;
    const bool by_run = m_out <= sm.m;
    float f_out = __builtin_amdgcn_exp2f(by_run ? fmaf(m_out, kLog2e, -sm.ref) : (m_out - top_safe) * kLog2e);
    const float to_top = __builtin_amdgcn_exp2f(fmaf(top_safe, kLog2e, -sm.ref)); // (2^ref over the exponential of the largest score: 1 over that)
    float f_run = by_run ? 1.f : __builtin_amdgcn_exp2f(-fmaf(top_safe, kLog2e, -sm.ref));
    const float inv = 1.0f / fmaf(quad_sum(sm.total_l), f_run, out_l[wave][n] * f_out);
    const float inv_top = by_run ? inv * to_top : inv; // relative to the exponential of the largest score
    f_run *= 1.f / TileWeights<T>::kScale;
#pragma unroll
    for (int c = 0; c < NB; ++c) {
        f32x4* at = reinterpret_cast<f32x4*>(part + n * PAD + TileCols<T, D>::at(c, gq));
        const f32x4 run = TileCols<T, D>::sums(sm.total, c);
        f32x4 o = *at;
#pragma unroll
        for (int x = 0; x < 4; ++x) o[x] = fmaf(run[x], f_run, o[x] * f_out) * inv;
        *at = o;
    }
    wave_lds_sync();
    f32x4* to = reinterpret_cast<f32x4*>(out + (size_t)row0 * D);
#pragma unroll
    for (int i = 0; i < kTileRows * D / 4 / kWave; ++i) {
        const int at = i * kWave + lane;
        to[at] = *reinterpret_cast<const f32x4*>(part + at / (D / 4) * PAD + at % (D / 4) * 4);
    }
    if (KEEP == kKeepScores && gq == 0) stats[row0 + n] = make_float2(top_safe, inv_top);
    if (KEEP == kKeepProbs) {
        __threadfence_block(); // (the wave's own scores, normalised in place)
        for (int r = 0; r < kTileRows; ++r) {
            const int4 row = extents[wave][r];
            const float top_r = __shfl(top_safe, r, kWave), inv_r = __shfl(inv_top, r, kWave);
            for (int slot = row.x + lane; slot < row.x + row.y; slot += kWave) probs[slot] = __expf(probs[slot] - top_r) * inv_r;
        }
    }
}

// Four tiles a workgroup (attention_wide_kernel, halves) or one?  fours: how many workgroups of four a head's longest one is worth
// (rode_hip_plans.tile_fours), 0 where the four lie apart or nothing is known.  The GPU has room for 1280, 1024 and 512 workgroups at a time
// (widths 32, 64 and 128; a wave per tile, the other kernel four): a few more than that take a second round nearly alone, and a wave per tile has to
// fill the GPU.  Width 32, where the values, not shared, are half of what is read, gains by it with short rows or after two rounds.  Time of four
// over that of one (64 and more random columns; none or few): 2700 masks of 1500 to 20 000 rows, windows of 128 to 640 and 0 to 96 random columns, 1 to 16 heads
//   width 128  375 workgroups 0.97 to 1.13; 0.83 to 1.04, 450 to 512 0.78 to 0.93; 0.67 to 0.92, 524 to 600 up to 1.16; 1.10, 700 0.90 to 1.08; 0.85 to
//              0.98, 750 0.84 to 1.02; 0.73 to 0.96, 1025 to 1300 0.81 to 0.98; 0.74 to 0.96
//   width 64   512 0.98 to 1.10; 0.76 to 1.14 (up to 300 nonzeros a row 1.04), 650 0.94 to 1.01; 0.92 to 0.97, 1000 0.80 to 0.93; 0.65 to 0.86, 1050 up to
//              1.12, 1150 1.06, 1250 0.94 to 1.02; 0.74 to 1.03, 2000 0.82 to 0.92; 0.65 to 0.87
//   width 32   1000 0.97 to 1.10; 0.75 to 1.04, 1300 up to 1.22, 1500 1.19, 2000 0.93 to 1.10; 0.72 to 1.06, 2500 0.93 to 0.97; 0.72 to 0.98
// One of those calls is more than 3 % slower than with a tile a workgroup (1.04).  From 512 workgroups on (1024 for width 32, 640 for rows of 600 of
// width 64), without a look at the rounds, 298 were, the most 1.22 (8352 rows of 578 and 96 random columns, four heads of 128: 152 -> 181 us).
//   fp32 (not taken), width 64 768: 104 -> 96, 640: 86 -> 92; 1024: 157 -> 152; width 128 1024: 349 -> 351; width 32 1024: 78 -> 78
inline bool tiles_in_fours(int d, int nheads, int M, int nnz, int fours)
{
    if (fours <= 0) return false;
    const long long worth = (long long)fours * nheads, quads = (row_tiles(M) + kWavesPerWg - 1) / kWavesPerWg;
    const long long wgs = quads * nheads > worth ? quads * nheads : worth;
    const auto rows_of = [&](int most) { return (long long)nnz < (long long)most * M; };
    if (d == 32) return wgs <= 1280 ? worth >= 900 && rows_of(220) : worth >= (rows_of(300) ? 1900 : 2450);
    if (d == 64) return wgs <= 1024 ? worth >= (rows_of(300) ? 512 : 640) : worth >= 1024 && wgs >= 1230;
    return wgs <= 512 ? worth >= 440 : worth >= 600 && wgs >= 740;
}

template <typename T, int D>
hipError_t launch_tiles(int nheads, int M, int N, int nnz, const int* row_ptr, const int* col, const float* val, const T* q, const T* k,
                        const T* v, float scale, float* out, float* probs, float2* stats, const int* plan, int plan_fours, hipStream_t stream)
{
    const int n_tiles = row_tiles(M);
    HeadStrides heads;
    heads.rows = (size_t)M * D, heads.cols = (size_t)N * D, heads.nnz = (size_t)nnz;
    if constexpr (sizeof(T) == 2) {
        if (tiles_in_fours(D, nheads, M, nnz, plan_fours)) {
            const long long items = (long long)((n_tiles + kWavesPerWg - 1) / kWavesPerWg) * nheads;
            const dim3 grid((unsigned)((items + kXcds - 1) / kXcds * kXcds));
            auto kernel = probs == nullptr ? attention_wide_kernel<T, D, kKeepNothing>
                          : stats != nullptr ? attention_wide_kernel<T, D, kKeepScores> : attention_wide_kernel<T, D, kKeepProbs>;
            kernel<<<grid, kWgThreads, 0, stream>>>(nheads, n_tiles, group_plan_tiles(plan, M), group_plan_runs(plan, M), row_ptr, col, val, q, k, v,
                                                    scale, out, probs, stats, heads);
            return hipGetLastError();
        }
    }
    const dim3 grid((n_tiles + kXcds - 1) / kXcds * kXcds, nheads);
    auto kernel = probs == nullptr ? attention_tile_kernel<T, D, kKeepNothing>
                  : stats != nullptr ? attention_tile_kernel<T, D, kKeepScores> : attention_tile_kernel<T, D, kKeepProbs>;
    kernel<<<grid, kWgThreads, 0, stream>>>(n_tiles, group_plan_tiles(plan, M), group_plan_runs(plan, M), row_ptr, col, val, q, k, v,
                                            scale, out, probs, stats, 2 * (size_t)N * D * sizeof(T) >= kOutsideFirstBytes, heads);
    return hipGetLastError();
}

} // namespace

// The tiles of a group plan (plan.groups, with plan.group_counts[3] > 0 of them); arguments as
// attention_launch.  One head's k or v must not exceed 4 GB (attention_tiles_fit).
template <typename T>
hipError_t attention_tiles_launch(int nheads, int M, int N, int nnz, int d, const int* row_ptr, const int* col, const float* val,
                                  const T* q, const T* k, const T* v, float scale, float* out, float* probs, float* row_stats,
                                  const int* plan, int plan_fours, hipStream_t stream)
{
    float2* stats = reinterpret_cast<float2*>(row_stats);
    switch (d) {
    case 32: return launch_tiles<T, 32>(nheads, M, N, nnz, row_ptr, col, val, q, k, v, scale, out, probs, stats, plan, plan_fours, stream);
    case 64: return launch_tiles<T, 64>(nheads, M, N, nnz, row_ptr, col, val, q, k, v, scale, out, probs, stats, plan, plan_fours, stream);
    case 128: return launch_tiles<T, 128>(nheads, M, N, nnz, row_ptr, col, val, q, k, v, scale, out, probs, stats, plan, plan_fours, stream);
    default: return hipErrorInvalidValue;
    }
}

template hipError_t attention_tiles_launch<float>(int, int, int, int, int, const int*, const int*, const float*, const float*, const float*,
                                                  const float*, float, float*, float*, float*, const int*, int, hipStream_t);
template hipError_t attention_tiles_launch<__half>(int, int, int, int, int, const int*, const int*, const float*, const __half*,
                                                   const __half*, const __half*, float, float*, float*, float*, const int*, int, hipStream_t);

} // namespace rode
