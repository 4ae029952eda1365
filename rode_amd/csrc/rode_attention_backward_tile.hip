// Gradient of sparse attention, row pass, for the tiles of 16 rows of a group plan, on the matrix
// cores (the contract of attention_backward_rows_kernel in rode_attention_backward.hip, which takes
// the rows of no tile):
//     dp = <g[r, :], v[col, :]>,  dz = scale * value * p * (dp - delta[r]),  dq[r, :] = sum of dz * k[col, :]
// and the pairs (p, dz) of every nonzero go to its slot in the transposed pattern.
//
// One workgroup per tile and head, as in the forward pass (rode_attention_tile.hip): its four waves take the
// columns of the run 16 or 32 at a time, in turn - dp^T = V G^T and dq^T += K^T dZ^T - and the
// nonzeros outside the run of four rows each; the partial sums of dq meet in LDS.  The score layout has
// the 16 rows of a tile in adjacent lanes, which is the order of a column in the transposed pattern:
// where every row holds a column its 16 pairs are 128 consecutive bytes, and one slot number is
// read for them instead of 16.  A non-finite row of k in the range that a row does not hold would reach it (0 * Inf)
// and shows as a non-finite sum: the tile is then computed again row by row.
//
// fp16 operands: g is scaled by the largest magnitude of its row and rounded to fp16 for dp, as in
// the other kernels; dz is split into two halves (TileWeights), times a power of two per row that
// follows the largest |dz| so far (the sums are rescaled when it moves, exactly).  The rounding of g is what decides
// there: dq is 2e-4 to 7e-4 off with and without tiles.
//
// Measured (16 384 rows, window 512 and 64 random columns, width 64, one head in fp32; the kernel's own time): 107 us with the
// nonzeros outside the run of one row after the other, 95 with those of four rows side by side (TileOutside); training step, us, the other two
// passes unchanged: fp32 250 -> 244, halves 172 -> 167, width 128 457 -> 422 and 316 -> 302; 20 000 rows of 300 + 96, width 64 430 -> 410.
// Bound by latency: 1.7 waves per SIMD (registers: two in fp32, three with halves of width 32, one with halves of width 128, whose LDS leaves
// one workgroup per CU) wait for memory 42 % of their time and for their turn 33 %; the vector ALUs issue 28 % of it, the address
// units are busy for 57 %, and 382 MB pass the L2s (4.3 TB/s; 190 MB of them values, scores, slots and pairs).  Tried before the
// nonzeros outside the run went side by side: three waves per SIMD (halves spill, step 0.250 ms instead of 0.21; fp32 0.282
// instead of 0.279).
#include "rode_tile.hpp"
#include "rode_units.hpp"
#include "rode_internal.hpp"

#include <type_traits>

namespace rode {

namespace {

typedef int i32x4_u __attribute__((ext_vector_type(4), aligned(4)));

// The power of two that keeps a row's dz within halves: the largest |dz| so far is below 2 * cap, and
// dz times factor() below 2^15.  (32-bit operands: none.)
template <typename T>
struct TileRange {
    __device__ __forceinline__ float factor() const { return 1.f; }
    __device__ __forceinline__ float back() const { return 1.f; }
    template <int N, int NB>
    __device__ __forceinline__ void step(const float (&)[N], f32x4 (&)[NB])
    {
    }
};
template <>
struct TileRange<__half> {
    float cap = 0x1p-112f;
    __device__ __forceinline__ float factor() const { return 0x1p14f / cap; }
    __device__ __forceinline__ float back() const { return cap * 0x1p-14f; }
    template <int N, int NB>
    __device__ __forceinline__ void step(const float (&dz)[N], f32x4 (&acc)[NB])
    {
        float top = fabsf(dz[0]);
#pragma unroll
        for (int j = 1; j < N; ++j) top = fmaxf(top, fabsf(dz[j]));
        top = quad_max(top);
        if (__any(top >= 2.f * cap)) {
            const float now = fmaxf(cap, __uint_as_float(__float_as_uint(top) & 0x7f800000u)); // (a non-finite one stays)
            const float corr = cap / now;
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[b] *= corr;
            cap = now;
        }
    }
};

template <typename T, int D>
__global__ void __launch_bounds__(kWgThreads, (tile_waves<T, D>()))
attention_backward_tile_kernel(int n_tiles, const RowTile* __restrict__ tiles, const int* __restrict__ runs,
                               const int* __restrict__ row_ptr, const int* __restrict__ col, const float* __restrict__ val,
                               const float* __restrict__ probs, const float2* __restrict__ stats, const float* __restrict__ g,
                               const float* __restrict__ out, const T* __restrict__ k, const T* __restrict__ v, float scale,
                               const int* __restrict__ t_slot, float* __restrict__ dq, float2* __restrict__ pz, HeadStrides heads)
{
    constexpr int NB = D / 16, PAD = D + 4, NT = tile_blocks<T>(), kStep = 16 * NT;
    constexpr bool kHalf = std::is_same<T, __half>::value;
    using VStage = TileStage<T, D, kAlong>;  // (v meets g along its elements, k is summed across)
    using KStage = TileStage<T, D, tile_columns<T>()>;
    // Per wave: staged rows of v and k, the values and what the forward pass kept of a step.  Then staging for the nonzeros outside
    // the runs, then the wave's partial sums and behind them the sums of its four rows outside their runs.
    constexpr int kPart = kTileRows * PAD, kStageFloats = 2 * VStage::kBytes / 4 + 2 * TileSquare<T>::kFloats;
    static_assert(kPart + kOutsideRows * PAD <= kStageFloats && 2 * kOutsideSteps * kWave <= kStageFloats, "what comes later fits");
    __shared__ __attribute__((aligned(16))) float shared[kWavesPerWg][kStageFloats];
    __shared__ int4 extents[kTileRows]; // (for the nonzeros outside the runs: not in registers until then)
    const int tile = xcd_logical_block(blockIdx.x, gridDim.x);
    if (tile >= n_tiles) return;
    const RowTile rt = tiles[tile];
    if (rt.hi <= rt.lo) return; // not a tile: other kernels have its rows
    probs = of_head(probs, heads.nnz), g = of_head(g, heads.rows), out = of_head(out, heads.rows);
    stats = of_head(stats, heads.rows / D);
    k = of_head(k, heads.cols), v = of_head(v, heads.cols), dq = of_head(dq, heads.rows), pz = of_head(pz, heads.nnz);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave; // (uniform: scalar registers)
    const int n = lane % 16, gq = lane / 16;
    const TileLane me = tile_lane(tile * kTileRows + n, row_ptr, runs);
    const int base = me.base();
    if (threadIdx.x < kTileRows) extents[threadIdx.x] = me.packed();
    const int steps = (rt.hi - rt.lo + kStep - 1) / kStep;
    u32x4* lds_v = reinterpret_cast<u32x4*>(shared[wave]);
    u32x4* lds_k = lds_v + VStage::kBytes / 16;
    f32x4* lds_w = reinterpret_cast<f32x4*>(lds_k + KStage::kBytes / 16);
    f32x4* lds_s = lds_w + TileSquare<T>::kFloats / 4;

    // the lane's row: its statistics, delta = <g, out>, and g as operand of the products
    const bool kept_scores = stats != nullptr;
    float stat_max = 0.f, stat_inv = 1.f;
    if (kept_scores) {
        const float2 s = stats[me.row];
        stat_max = s.x, stat_inv = s.y;
    }
    auto prob_of = [&](float kept, float top, float inv) __attribute__((always_inline)) {
        return kept_scores ? __expf(kept - top) * inv : kept;
    };
    TileRow<T, D> g_row;
    float delta = 0.f, g_scale = 1.f, g_inv = 1.f;
    {
        constexpr int kChunks = TileRow<T, D>::kChunks, kElems = 16 / (int)sizeof(T);
        f32x4 raw[kChunks][kElems / 4];
        float big = 0.f;
#pragma unroll
        for (int i = 0; i < kChunks; ++i)
#pragma unroll
            for (int h = 0; h < kElems / 4; ++h) {
                const size_t at = (size_t)me.row * D + 4 * kElems * i + kElems * gq + 4 * h;
                raw[i][h] = *reinterpret_cast<const f32x4*>(g + at);
                const f32x4 o = *reinterpret_cast<const f32x4*>(out + at);
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    delta = fmaf(raw[i][h][x], o[x], delta);
                    big = fmaxf(big, fabsf(raw[i][h][x]));
                }
            }
        delta = quad_sum(delta);
        if constexpr (kHalf) {
            g_scale = quad_max(big);
            g_inv = g_scale > 0.f ? 1.0f / g_scale : 0.f;
#pragma unroll
            for (int i = 0; i < kChunks; ++i)
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const __half2 h2 = __floats2half2_rn(raw[i][x / 2][2 * (x % 2)] * g_inv, raw[i][x / 2][2 * (x % 2) + 1] * g_inv);
                    g_row.c[i][x] = *reinterpret_cast<const uint32_t*>(&h2);
                }
        } else {
#pragma unroll
            for (int i = 0; i < kChunks; ++i) g_row.c[i] = __builtin_bit_cast(u32x4, raw[i][0]);
        }
    }

    f32x4 acc[NB];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = kNothing;
    };
    clear();
    TileRange<T> range;

    // This wave's four rows without the nonzeros of their runs (or, `whole`, with them), 64 of each row at a time: 16 lanes
    // have a row's nonzeros, LPR lanes read a dense row, 16 bytes each, every lane group the rows of its own LPR
    // nonzeros.  The rows of v of all 64 first, then those of k.
    auto rows_outside = [&](bool whole) __attribute__((always_inline)) {
        using Out = TileOutside<T, D>;
        constexpr int VEC = Out::kVec, LPR = Out::kLpr, RPG = Out::kRows, QUADS = Out::kQuads, S = kOutsideSteps;
        const int ls = lane % LPR, group = lane / LPR;
        const unsigned lane_at = ls * 16u; // (an operand of a tile is at most 4 GB: 32-bit offsets)
        const char* k_bytes = reinterpret_cast<const char*>(k);
        const char* v_bytes = reinterpret_cast<const char*>(v);
        unsigned* my_at = reinterpret_cast<unsigned*>(shared[wave]); // (the step's staging is free)
        float* my_z = shared[wave] + S * kWave;
        const Out of(extents, wave, lane, whole);
        const float row_max = __shfl(stat_max, of.mine, kWave), row_inv = __shfl(stat_inv, of.mine, kWave);
        const float row_delta = __shfl(delta, of.mine, kWave), row_scale = __shfl(g_scale, of.mine, kWave);
        typename DotVec<T>::Reg a[RPG][DotVec<T>::kRegs];
#pragma unroll
        for (int i = 0; i < RPG; ++i) {
            const float* g_at = g + (size_t)(tile * kTileRows + of.row(i)) * D + ls * VEC;
            f32x4 x[VEC / 4];
#pragma unroll
            for (int h = 0; h < VEC / 4; ++h) x[h] = *reinterpret_cast<const f32x4*>(g_at + 4 * h);
            if constexpr (kHalf) {
                const float row_back = __shfl(g_inv, of.row(i), kWave);
#pragma unroll
                for (int y = 0; y < 4; ++y) {
                    const __half2 h2 = __floats2half2_rn(x[y / 2][2 * (y % 2)] * row_back, x[y / 2][2 * (y % 2) + 1] * row_back);
                    a[i][y] = *reinterpret_cast<const uint32_t*>(&h2);
                }
            } else {
#pragma unroll
                for (int y = 0; y < 4; ++y) a[i][y] = x[0][y];
            }
        }
        float sum[RPG][VEC];
#pragma unroll
        for (int i = 0; i < RPG; ++i)
#pragma unroll
            for (int x = 0; x < VEC; ++x) sum[i][x] = 0.f;
#pragma unroll 1
        for (int off = 0; off < of.most; off += 16 * S) {
            float w[S], kept[S];
            int to[S];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                int c = 0;
                w[s] = kept[s] = 0.f;
                to[s] = 0;
                if (off + 16 * s < of.cnt) { // (lanes past the end repeat the last nonzero with weight 0)
                    const int idx = of.slot(off + 16 * s + lane % 16);
                    c = col[idx], to[s] = t_slot[idx], w[s] = val[idx], kept[s] = probs[idx];
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
                        uint4 v_part[QUADS][4];
#pragma unroll
                        for (int u = 0; u < QUADS; ++u) {
                            const u32x4 o = *reinterpret_cast<const u32x4*>(my_at + s * kWave + group * LPR + 4 * (i * QUADS + u));
#pragma unroll
                            for (int j = 0; j < 4; ++j) v_part[u][j] = *reinterpret_cast<const uint4*>(v_bytes + (o[j] + lane_at));
                        }
#pragma unroll
                        for (int u = 0; u < QUADS; ++u) {
                            float part[4];
#pragma unroll
                            for (int j = 0; j < 4; ++j) part[j] = DotVec<T>::dot_raw(a[i], v_part[u][j], 0.f);
                            const float dot = sddmm_quad_reduce<LPR>(part, ls);
                            if ((ls >> 2) == i * QUADS + u) d = dot;
                        }
                    }
                const bool live = off + 16 * s + lane % 16 < of.cnt;
                const float p = prob_of(kept[s], row_max, row_inv), dz = live ? scale * w[s] * p * (d * row_scale - row_delta) : 0.f;
                if (live) pz[to[s]] = make_float2(p, dz);
                my_z[s * kWave + lane] = dz;
            }
            wave_lds_sync();
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < RPG; ++i)
                    if (off + 16 * s < of.cnt_of[i]) Out::add(k_bytes, lane_at, my_at + s * kWave, my_z + s * kWave, group * LPR + 4 * i * QUADS, sum[i]);
            wave_lds_sync();
        }
        of.store(sum, shared[wave] + kPart, PAD, lane);
    };

    // a step's columns of the run, on their way
    VStage v_rows;
    KStage k_rows;
    f32x4 w_rows[NT], s_rows[NT];
    i32x4_u to_first[NT], to_last[NT]; // slots in the transposed pattern: of the tile's first and last row
    // (the row and the four columns that this lane fetches values of: TileSquare)
    const int f_a = __shfl(me.a, lane / 4, kWave), f_end = f_a + __shfl(me.len, lane / 4, kWave), f_base = __shfl(base, lane / 4, kWave);
    const int base_first = __builtin_amdgcn_readlane(base, 0), base_last = __builtin_amdgcn_readlane(base, kTileRows - 1);
    auto inside = [&](int c0) { return c0 >= rt.core_lo && c0 + kStep <= rt.core_hi; }; // does every row hold every one of them?
    auto fetch = [&](int c0) __attribute__((always_inline)) {
        const bool in = inside(c0);
        v_rows.load(v + (size_t)c0 * D, rt.hi - 1 - c0, in, lane); // (columns past the range repeat its last)
        k_rows.load(k + (size_t)c0 * D, rt.hi - 1 - c0, in, lane);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int c = c0 + 16 * t + lane % 4 * 4;
            if (in) {
                w_rows[t] = *reinterpret_cast<const f32x4_u*>(val + f_base + c);
                s_rows[t] = *reinterpret_cast<const f32x4_u*>(probs + f_base + c);
                to_first[t] = *reinterpret_cast<const i32x4_u*>(t_slot + base_first + c0 + 16 * t + 4 * gq);
                to_last[t] = *reinterpret_cast<const i32x4_u*>(t_slot + base_last + c0 + 16 * t + 4 * gq);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool held = c + i >= f_a && c + i < f_end;
                    w_rows[t][i] = held ? val[f_base + c + i] : 0.f;
                    s_rows[t][i] = held ? probs[f_base + c + i] : 0.f;
                }
            }
        }
    };
    auto run_columns = [&]() __attribute__((always_inline)) {
        if (wave < steps) fetch(rt.lo + wave * kStep);
        for (int it = wave; it < steps; it += kWavesPerWg) {
            const int c0 = rt.lo + it * kStep;
            const bool in = inside(c0);
            v_rows.store(lds_v, lane);
            k_rows.store(lds_k, lane);
            int to[NT][4];
            bool apart = !in; // (a column that a row holds twice: the rows' slots are not consecutive)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                TileSquare<T>::in_order(lds_w, t, lane) = w_rows[t];
                TileSquare<T>::in_order(lds_s, t, lane) = s_rows[t];
                if (in) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        to[t][i] = to_first[t][i] + n;
                        apart = apart || to_last[t][i] - to_first[t][i] != kTileRows - 1;
                    }
                }
            }
            if (__any(apart)) {
#pragma unroll
                for (int j = 0; j < 4 * NT; ++j) {
                    const int c = c0 + 16 * (j / 4) + 4 * gq + j % 4;
                    to[j / 4][j % 4] = c >= me.a && c < me.a + me.len ? t_slot[base + c] : -1;
                }
            }
            wave_lds_sync();
            if (it + kWavesPerWg < steps) fetch(c0 + kWavesPerWg * kStep); // (in flight during this step)
            float dz[4 * NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                TileRow<T, D> v_row;
                VStage::read(lds_v, t, lane, v_row);
                const f32x4 dp = mma_rows<T, D>(v_row, g_row), w = TileSquare<T>::as_scores(lds_w, t, lane), kept = TileSquare<T>::as_scores(lds_s, t, lane);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = prob_of(kept[i], stat_max, stat_inv);
                    const float z = scale * w[i] * p * (dp[i] * g_scale - delta);
                    dz[4 * t + i] = to[t][i] >= 0 ? z : 0.f;
                    if (to[t][i] >= 0) pz[to[t][i]] = make_float2(p, z);
                }
            }
            range.step(dz, acc);
            TileWeights<T> weights;
            weights.set(dz, range.factor());
            TileCols<T, D> k_cols;
            k_cols.load(lds_k, lane);
            k_cols.accumulate(weights, acc);
            wave_lds_sync();
        }
    };

    run_columns();
    const bool again = __syncthreads_or(!all_finite<NB>(acc));
    if (again) clear();
    rows_outside(again);

    float* part = shared[wave];
    const float back = range.back();
#pragma unroll
    for (int c = 0; c < NB; ++c) {
        const f32x4 sums = TileCols<T, D>::sums(acc, c);
        *reinterpret_cast<f32x4*>(part + n * PAD + TileCols<T, D>::at(c, gq)) = again ? kNothing : sums * back;
    }
    __syncthreads();
    const int r = threadIdx.x / 16, e0 = threadIdx.x % 16 * NB;
    float o[NB];
#pragma unroll
    for (int x = 0; x < NB; ++x) {
        o[x] = shared[r / kOutsideRows][kPart + r % kOutsideRows * PAD + e0 + x];
#pragma unroll
        for (int w = 0; w < kWavesPerWg; ++w) o[x] += shared[w][r * PAD + e0 + x];
    }
#pragma unroll
    for (int x = 0; x < NB; x += 2)
        *reinterpret_cast<float2*>(dq + (size_t)(tile * kTileRows + r) * D + e0 + x) = make_float2(o[x], o[x + 1]);
}

template <typename T, int D>
hipError_t launch_tiles(int nheads, int M, HeadStrides heads, const int* row_ptr, const int* col, const float* val, const float* probs,
                        const float2* stats, const float* g, const float* out, const T* k, const T* v, float scale, const int* t_slot,
                        float* dq, float2* pz, const int* plan, hipStream_t stream)
{
    const int n_tiles = row_tiles(M);
    const dim3 grid((n_tiles + kXcds - 1) / kXcds * kXcds, nheads);
    attention_backward_tile_kernel<T, D><<<grid, kWgThreads, 0, stream>>>(n_tiles, group_plan_tiles(plan, M), group_plan_runs(plan, M), row_ptr,
                                                                          col, val, probs, stats, g, out, k, v, scale, t_slot, dq, pz, heads);
    return hipGetLastError();
}

} // namespace

// The tiles of a group plan (plan: with tiles); arguments as attention_backward_rows_launch.  One head's k or v
// must not exceed 4 GB (attention_tiles_fit).
template <typename T>
hipError_t attention_backward_tiles_launch(int nheads, int M, int N, int nnz, int d, const int* row_ptr, const int* col, const float* val,
                                           const float* probs, const float* row_stats, const float* g, const float* out, const T* k,
                                           const T* v, float scale, const int* t_slot, float* dq, float* pz, const int* plan,
                                           hipStream_t stream)
{
    HeadStrides heads;
    heads.rows = (size_t)M * d, heads.cols = (size_t)N * d, heads.nnz = (size_t)nnz;
    const float2* stats = reinterpret_cast<const float2*>(row_stats);
    float2* pairs = reinterpret_cast<float2*>(pz);
    switch (d) {
    case 32: return launch_tiles<T, 32>(nheads, M, heads, row_ptr, col, val, probs, stats, g, out, k, v, scale, t_slot, dq, pairs, plan, stream);
    case 64: return launch_tiles<T, 64>(nheads, M, heads, row_ptr, col, val, probs, stats, g, out, k, v, scale, t_slot, dq, pairs, plan, stream);
    case 128: return launch_tiles<T, 128>(nheads, M, heads, row_ptr, col, val, probs, stats, g, out, k, v, scale, t_slot, dq, pairs, plan, stream);
    default: return hipErrorInvalidValue;
    }
}

template hipError_t attention_backward_tiles_launch<float>(int, int, int, int, int, const int*, const int*, const float*, const float*,
                                                           const float*, const float*, const float*, const float*, const float*, float,
                                                           const int*, float*, float*, const int*, hipStream_t);
template hipError_t attention_backward_tiles_launch<__half>(int, int, int, int, int, const int*, const int*, const float*, const float*,
                                                            const float*, const float*, const float*, const __half*, const __half*, float,
                                                            const int*, float*, float*, const int*, hipStream_t);

} // namespace rode
