// Gradient of sparse attention, column pass, for the tiles of 16 rows of a group plan of the transposed pattern
// (16 adjacent columns of the mask whose rows share a run), on the matrix cores (the contract of
// attention_backward_cols_kernel in rode_attention_backward.hip, which takes the rows of no tile):
//     dv[c, :] = sum of p * g[row, :],  dk[c, :] = sum of dz * q[row, :]
// over the nonzeros of column c, the pairs (p, dz) in the order of the transposed pattern.
//
// One workgroup per tile and head, as in the other tile kernels (rode_tile.hpp has the layouts): its four waves take
// 16 rows of the run at a time, in turn - dv^T += G^T P^T and dk^T += Q^T dZ^T, every row of g and of q loaded once for 16
// columns - and then the nonzeros outside the run of four columns each, 16 of each column at a time: 64 of every column are
// looked up together, their rows of g first and then those of q (half the rows at a time are wanted, and the columns' rows
// ascend, so that more of them are found in L2).  The waves' sums meet in LDS.
// Both products are 32-bit ones whatever q is (halves are widened on their way out of LDS, exactly): the pairs keep
// their 32 bits.  A non-finite row of g or q in the range that a column does not hold would reach it (0 * Inf) and
// shows as a non-finite sum: the tile is then computed again column by column.
//
// Measured (16 384 rows, window 512 and 64 random columns): the pass in fp32, width 64, 89 us with four columns at a time on the
// vector ALUs, 69 here (along the run 38, 32-bit matrix products and the pairs; outside it 31; 346 MB past the L2s, the vector
// ALUs issue 24 % of the time; 2.9 waves per SIMD wait for memory 29 % of theirs and for their turn 57 %).  Training step, one
// head, fp32 widths 32 / 64 / 128: 159 -> 145, 274 -> 253, 550 -> 491 us; halves 138 -> 127, 193 -> 175, 360 -> 328; four heads of
// width 64 1079 -> 985, halves 827 -> 745; without random columns 627 -> 521, halves 539 -> 435.  On the way, the pass in fp32: nonzeros
// outside the run of one column after the other 80; of four columns, g and q together 75; outside first 76 (spills);
// every other wave in that order 81.
#include "rode_tile.hpp"
#include "rode_units.hpp"
#include "rode_internal.hpp"

namespace rode {

namespace {

typedef float f32x4_pair __attribute__((ext_vector_type(4), aligned(8))); // two pairs at any pair's address

constexpr int kColsStep = 16;    // rows of the run that a wave takes at a time
constexpr int kColsOutside = 4;  // times 16 nonzeros of every column outside the run

// Waves per SIMD that the registers leave room for: as many as LDS does (a workgroup of width 64 takes 40 KB, so that the 1024 tiles
// of 16 384 columns are all resident; with three per SIMD a third of them would come after the others).
template <int D>
constexpr int cols_tile_waves()
{
    return D == 128 ? 2 : 4;
}

template <typename T, int D>
__global__ void __launch_bounds__(kWgThreads, (cols_tile_waves<D>()))
attention_backward_cols_tile_kernel(int n_tiles, const RowTile* __restrict__ tiles, const int* __restrict__ runs,
                                    const int* __restrict__ t_row_ptr, const int* __restrict__ t_col, const float2* __restrict__ pz,
                                    const float* __restrict__ g, const T* __restrict__ q, float* __restrict__ dk,
                                    float* __restrict__ dv, HeadStrides heads)
{
    constexpr int NB = D / 16;
    using GStage = TileStage<float, D, kAcross, kColsStep>;
    using QStage = TileStage<T, D, kAcross, kColsStep>;
    using Square = TileSquare<float>;
    // Per wave: staged rows of g and q and the step's p and dz; then the wave's sums of dv and dk in the same place, and behind
    // them rows and weights of nonzeros outside the run.  (Width 64: 40 KB, four workgroups per CU.)
    constexpr int kPart = kTileRows * D, kStaged = (GStage::kBytes + QStage::kBytes) / 4 + 2 * Square::kFloats;
    constexpr int kFloats = kStaged > 2 * kPart + 2 * kColsOutside * kWave ? kStaged : 2 * kPart + 2 * kColsOutside * kWave, kOutside = 2 * kPart;
    __shared__ __attribute__((aligned(16))) float shared[kWavesPerWg][kFloats];
    const int tile = xcd_logical_block(blockIdx.x, gridDim.x);
    if (tile >= n_tiles) return;
    const RowTile rt = tiles[tile];
    if (rt.hi <= rt.lo) return; // not a tile: other kernels have its rows
    pz = of_head(pz, heads.nnz), g = of_head(g, heads.rows), q = of_head(q, heads.rows);
    dk = of_head(dk, heads.cols), dv = of_head(dv, heads.cols);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave; // (uniform: scalar registers)
    const int n = lane % 16, gq = lane / 16;
    const TileLane me = tile_lane(tile * kTileRows + n, t_row_ptr, runs);
    const int steps = (rt.hi - rt.lo + kColsStep - 1) / kColsStep;
    // element e of a sum of column c of the tile (rotated: the lanes of different columns in banks of their own)
    auto place = [](int c, int e) { return c * D + ((e + 4 * c) & (D - 1)); };
    u32x4* lds_g = reinterpret_cast<u32x4*>(shared[wave]);
    u32x4* lds_q = lds_g + GStage::kBytes / 16;
    f32x4* lds_p = reinterpret_cast<f32x4*>(lds_q + QStage::kBytes / 16);
    f32x4* lds_z = lds_p + Square::kFloats / 4;

    f32x4 acc_v[NB], acc_k[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc_v[b] = acc_k[b] = kNothing;

    // a step's rows and pairs, on their way (this lane: the four pairs of row lane / 4 from 4 * (lane % 4) on: TileSquare)
    GStage g_rows;
    QStage q_rows;
    f32x4 pairs[2];
    const int f_a = __shfl(me.a, lane / 4, kWave), f_end = f_a + __shfl(me.len, lane / 4, kWave), f_base = __shfl(me.base(), lane / 4, kWave);
    auto fetch = [&](int r0) __attribute__((always_inline)) {
        const bool in = r0 >= rt.core_lo && r0 + kColsStep <= rt.core_hi; // does every column hold every one of the rows?
        g_rows.load(g + (size_t)r0 * D, rt.hi - 1 - r0, in, lane); // (rows past the range repeat its last)
        q_rows.load(q + (size_t)r0 * D, rt.hi - 1 - r0, in, lane);
        const int r = r0 + lane % 4 * 4;
        if (in) {
#pragma unroll
            for (int h = 0; h < 2; ++h) pairs[h] = *reinterpret_cast<const f32x4_pair*>(pz + (f_base + r + 2 * h));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool held = r + i >= f_a && r + i < f_end;
                const float2 x = held ? pz[f_base + r + i] : make_float2(0.f, 0.f);
                pairs[i / 2][2 * (i % 2)] = x.x, pairs[i / 2][2 * (i % 2) + 1] = x.y;
            }
        }
    };
    auto run_rows = [&]() __attribute__((always_inline)) {
        if (wave < steps) fetch(rt.lo + wave * kColsStep);
        for (int it = wave; it < steps; it += kWavesPerWg) {
            g_rows.store(lds_g, lane);
            q_rows.store(lds_q, lane);
            Square::in_order(lds_p, 0, lane) = f32x4{pairs[0][0], pairs[0][2], pairs[1][0], pairs[1][2]};
            Square::in_order(lds_z, 0, lane) = f32x4{pairs[0][1], pairs[0][3], pairs[1][1], pairs[1][3]};
            wave_lds_sync();
            if (it + kWavesPerWg < steps) fetch(rt.lo + (it + kWavesPerWg) * kColsStep); // (in flight during this step)
            TileCols<float, D> cols;
            TileWeights<float> weights;
            const f32x4 p = Square::as_scores(lds_p, 0, lane), z = Square::as_scores(lds_z, 0, lane);
#pragma unroll
            for (int j = 0; j < 4; ++j) cols.load(j, GStage::across(lds_g, 4 * gq + j, n)), weights.p[j] = p[j];
            cols.accumulate(weights, acc_v);
#pragma unroll
            for (int j = 0; j < 4; ++j) cols.load(j, QStage::across(lds_q, 4 * gq + j, n)), weights.p[j] = z[j];
            cols.accumulate(weights, acc_k);
            wave_lds_sync();
        }
    };

    // This wave's four columns without the nonzeros of their runs (or, `whole`, with them), 16 of each at a time: LPR lanes
    // read a dense row, 16 bytes of g each, every lane group the rows of its own LPR nonzeros.
    float* part = shared[wave];
    auto rows_outside = [&](bool whole) __attribute__((always_inline)) {
        constexpr int LPR = D / 4, R = kTileRows / kWavesPerWg, kSteps = kColsOutside, RPG = LPR > 16 ? LPR / 16 : 1; // (columns of a lane group)
        static_assert(R == 4, "16 lanes per column");
        const int ls = lane % LPR, group = lane / LPR;
        const float* g_lane = g + ls * 4;
        const T* q_lane = q + ls * 4;
        int* my_r = reinterpret_cast<int*>(shared[wave] + kOutside);
        float* my_x = shared[wave] + kOutside + kSteps * kWave; // (p, then dz)
        const int mine = R * wave + lane / 16; // this lane's column
        const int first = __shfl(me.s, mine, kWave), split = __shfl(me.pos, mine, kWave), jump = whole ? 0 : __shfl(me.len, mine, kWave);
        const int cnt = __shfl(me.e, mine, kWave) - first - jump;
        int most = 0, cnt_of[RPG]; // (of all four; of this lane group's)
#pragma unroll
        for (int i = 0; i < R; ++i) most = max(most, __builtin_amdgcn_readlane(cnt, 16 * i));
#pragma unroll
        for (int i = 0; i < RPG; ++i) cnt_of[i] = RPG == 1 ? cnt - group * LPR % 16 : __shfl(cnt, group * LPR + 16 * i, kWave);
        float sum[2][RPG][4];
#pragma unroll
        for (int i = 0; i < RPG; ++i)
#pragma unroll
            for (int y = 0; y < 4; ++y) sum[0][i][y] = sum[1][i][y] = 0.f;
#pragma unroll 1
        for (int off = 0; off < most; off += 16 * kSteps) {
            int r[kSteps];
            float2 x[kSteps];
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                const int slot = off + 16 * s + lane % 16, at = min(slot, cnt - 1); // (past the end: the last nonzero with weights 0)
                r[s] = 0, x[s] = make_float2(0.f, 0.f);
                if (off + 16 * s < cnt) {
                    const int idx = first + at + (at >= split ? jump : 0);
                    r[s] = t_col[idx];
                    if (slot < cnt) x[s] = pz[idx];
                }
            }
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                my_r[s * kWave + lane] = r[s];
                my_x[s * kWave + lane] = x[s].x;
            }
            wave_lds_sync();
            // all rows of g, then all of q
            auto gather = [&](auto* dense_lane, int h) __attribute__((always_inline)) {
#pragma unroll 1
                for (int s = 0; s < kSteps; ++s)
#pragma unroll
                    for (int i = 0; i < RPG; ++i)
                        if (off + 16 * s < cnt_of[i]) {
                            constexpr int QUADS = LPR / 4 / RPG;
                            const int at = s * kWave + group * LPR + i * QUADS * 4;
                            float step[4] = {0.f, 0.f, 0.f, 0.f};
                            float b[QUADS][4][4], w[QUADS][4];
#pragma unroll
                            for (int u = 0; u < QUADS; ++u) {
                                const int4 r4 = *reinterpret_cast<const int4*>(my_r + at + 4 * u);
                                const int row[4] = {r4.x, r4.y, r4.z, r4.w};
                                load_quad(my_x + at + 4 * u, w[u]);
#pragma unroll
                                for (int t = 0; t < 4; ++t) load4(dense_lane + (size_t)row[t] * D, b[u][t]);
                            }
#pragma unroll
                            for (int u = 0; u < QUADS; ++u)
#pragma unroll
                                for (int t = 0; t < 4; ++t)
#pragma unroll
                                    for (int y = 0; y < 4; ++y) step[y] = fmaf(w[u][t], b[u][t][y], step[y]);
#pragma unroll
                            for (int y = 0; y < 4; ++y) sum[h][i][y] += step[y];
                        }
            };
            gather(g_lane, 0);
            wave_lds_sync();
#pragma unroll
            for (int s = 0; s < kSteps; ++s) my_x[s * kWave + lane] = x[s].y;
            wave_lds_sync();
            gather(q_lane, 1);
            wave_lds_sync();
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < RPG; ++i) {
                const int c = RPG == 1 ? mine : R * wave + group * RPG + i;
                f32x4 total = {sum[h][i][0], sum[h][i][1], sum[h][i][2], sum[h][i][3]};
                if constexpr (LPR < 16) { // (several lane groups have a column)
#pragma unroll
                    for (int y = 0; y < 4; ++y) total[y] = butterfly_sum<LPR, 16>(total[y]);
                }
                if (LPR >= 16 || group % (16 / (LPR < 16 ? LPR : 16)) == 0) {
                    f32x4* at = reinterpret_cast<f32x4*>(part + h * kPart + place(c, ls * 4));
                    *at = *at + total;
                }
            }
    };

    run_rows();
    float* flag = part + kOutside; // are the wave's sums finite?
    const bool finite = !__any(!(all_finite<NB>(acc_v) && all_finite<NB>(acc_k)));
    if (lane == 0) *flag = finite ? 0.f : 1.f;
    __syncthreads();
    bool again = false;
#pragma unroll
    for (int w = 0; w < kWavesPerWg; ++w) again = again || shared[w][kOutside] != 0.f;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < D / 4; ++e) {
        part[place(n, (D / 4) * gq + e)] = again ? 0.f : acc_v[e % NB][e / NB];
        part[kPart + place(n, (D / 4) * gq + e)] = again ? 0.f : acc_k[e % NB][e / NB];
    }
    wave_lds_sync();
    rows_outside(again);
    __syncthreads();
    const int c = threadIdx.x / 16, e0 = threadIdx.x % 16 * NB;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float o[NB];
#pragma unroll
        for (int x = 0; x < NB; ++x) {
            o[x] = shared[0][h * kPart + place(c, e0 + x)];
#pragma unroll
            for (int w = 1; w < kWavesPerWg; ++w) o[x] += shared[w][h * kPart + place(c, e0 + x)];
        }
        float* to = (h == 0 ? dv : dk) + (size_t)(tile * kTileRows + c) * D + e0;
#pragma unroll
        for (int x = 0; x < NB; x += 2) *reinterpret_cast<float2*>(to + x) = make_float2(o[x], o[x + 1]);
    }
}

template <typename T, int D>
hipError_t launch_tiles(int nheads, int N, HeadStrides heads, const int* t_row_ptr, const int* t_col, const float2* pz, const float* g,
                        const T* q, float* dk, float* dv, const int* plan, hipStream_t stream)
{
    const int n_tiles = row_tiles(N);
    const dim3 grid((n_tiles + kXcds - 1) / kXcds * kXcds, nheads);
    attention_backward_cols_tile_kernel<T, D><<<grid, kWgThreads, 0, stream>>>(n_tiles, group_plan_tiles(plan, N), group_plan_runs(plan, N),
                                                                               t_row_ptr, t_col, pz, g, q, dk, dv, heads);
    return hipGetLastError();
}

} // namespace

// The tiles of a group plan of the transposed pattern (plan: with tiles); arguments as attention_backward_cols_launch.
template <typename T>
hipError_t attention_backward_cols_tiles_launch(int nheads, int M, int N, int nnz, int d, const int* t_row_ptr, const int* t_col,
                                                const float* pz, const float* g, const T* q, float* dk, float* dv, const int* plan,
                                                hipStream_t stream)
{
    HeadStrides heads;
    heads.rows = (size_t)M * d, heads.cols = (size_t)N * d, heads.nnz = (size_t)nnz;
    const float2* pairs = reinterpret_cast<const float2*>(pz);
    switch (d) {
    case 32: return launch_tiles<T, 32>(nheads, N, heads, t_row_ptr, t_col, pairs, g, q, dk, dv, plan, stream);
    case 64: return launch_tiles<T, 64>(nheads, N, heads, t_row_ptr, t_col, pairs, g, q, dk, dv, plan, stream);
    case 128: return launch_tiles<T, 128>(nheads, N, heads, t_row_ptr, t_col, pairs, g, q, dk, dv, plan, stream);
    default: return hipErrorInvalidValue;
    }
}

template hipError_t attention_backward_cols_tiles_launch<float>(int, int, int, int, int, const int*, const int*, const float*, const float*,
                                                                const float*, float*, float*, const int*, hipStream_t);
template hipError_t attention_backward_cols_tiles_launch<__half>(int, int, int, int, int, const int*, const int*, const float*, const float*,
                                                                 const __half*, float*, float*, const int*, hipStream_t);

} // namespace rode
