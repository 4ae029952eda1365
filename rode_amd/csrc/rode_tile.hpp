// Tiles of 16 rows on the matrix cores: what the attention kernels share (forward:
// rode_attention_tile.hip).  A tile is four adjacent groups of a group plan whose runs of
// consecutive columns overlap for the most part (RowTile, rode_items.hpp): along those columns
// scores and weighted sums are dense 16 x 16 products, and every dense row loaded serves 16 rows.
//
// Lane layouts (n = lane % 16, gq = lane / 16; MFMA 16x16: operand A has m = lane % 16, operand B
// has n = lane % 16, the result has column n = lane % 16 and rows 4 gq .. 4 gq + 3 in its four
// registers; which k a lane's elements stand for may be chosen freely, the same for A and B):
//   * a dense row as operand along its elements ("chunks"): 16 bytes at every 64 ch + 16 gq.
//     Adjacent lanes then want different rows, which the vector memory pipe serves one lane per clock
//     (64 clocks a load; 16 when every four adjacent lanes ask for 64 consecutive bytes): 32 rows are
//     loaded in order and re-arranged in LDS (TileStage);
//   * scores come out transposed, S^T = K Q^T: lane (n, gq) has row n of the tile and the four
//     columns 4 gq + i of a 16-column block.  A row's statistics are then one number per lane, its
//     values and scores are 16 consecutive bytes in memory, and the probabilities are operand B of
//     the next product as they are (k slot (gq, t, i) stands for column 16 t + 4 gq + i);
//   * the weighted sum too: O^T = V^T P^T.  32-bit operands: operand A has a lane per 16th of the elements, lane m
//     loads the D / 16 consecutive elements from (D / 16) m of each of its four columns' rows
//     (16 lanes, a whole row), product nb takes element nb of each, and lane (n, gq) ends up with the
//     D / 4 consecutive elements from (D / 4) gq of row n.  Halves: LDS transposes on the way out (TileCols), product nb
//     takes elements 16 nb .. 16 nb + 15, and lane (n, gq) ends up with elements 16 nb + 4 gq + i.  TileCols::sums and at
//     say which, four consecutive elements at a time.
#pragma once
#include "rode_items.hpp"
#include "rode_device.hpp"

namespace rode {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4))); // four consecutive floats at any 4-byte address

// 16-column blocks that a wave takes at a time: what one weighted-sum product of 16-bit operands
// contracts over (32 columns); 32-bit operands take 16 (the same bytes in LDS and registers).
template <typename T>
constexpr int tile_blocks()
{
    return sizeof(T) == 2 ? 2 : 1;
}

// Waves per SIMD that the compiler has to leave registers for, in the forward and the row pass.  It is told only where it would
// otherwise miss by a few the number that LDS allows (row pass in fp32: width 32 136 registers instead of 128, width 128 289
// instead of 256; forward of width 128 with scores 258): a kernel that is told keeps the accumulators out of the second half of the
// registers, and with halves that cost more than it gave (forward, two heads of width 32 / 64 / 128: 39.6, 59.8, 125 us left
// alone, 40.8, 63.1, 129 told; measured with the nonzeros outside the runs one row after the other).  The row pass with halves of width
// 128 has one workgroup per CU whatever it is told: its 82 432 bytes of LDS are 512 more than half of what there is; the forward of
// that width, 260 registers by itself, is told two (attention_tile_kernel).
template <typename T, int D>
constexpr int tile_waves()
{
    return sizeof(T) == 2 || D == 64 ? 1 : D == 32 ? 4 : 2;
}

constexpr float kLog2e = 1.44269504088896340736f;

// Sum and maximum over the four lanes of a row (lanes 16 and 32 apart).
__device__ __forceinline__ float quad_sum(float v) { return butterfly_sum<16, kWave>(v); }
__device__ __forceinline__ float quad_max(float v) { return butterfly_max<16, kWave>(v); }

// ---- chunks: a dense row along its elements ------------------------------------------------
template <typename T, int D>
struct TileRow {
    static constexpr int kChunks = D * (int)sizeof(T) / 64;
    u32x4 c[kChunks];
    __device__ __forceinline__ void load(const T* row, int gq)
    {
#pragma unroll
        for (int i = 0; i < kChunks; ++i) c[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(row) + 64 * i + 16 * gq);
    }
};

constexpr f32x4 kNothing = {0.f, 0.f, 0.f, 0.f};

// Rows of a (16 of them, m = lane % 16) times rows of b (n = lane % 16).  Every instruction has a sum of its own, and
// the sums meet in a tree, as the lanes' do in the row kernels: along one chain of D products the rounding errors are up
// to 2.8 times theirs (rms over the square root of D, fp32, D = 32 / 64 / 128: 1.03e-7, 1.44e-7, 2.04e-7 along a chain, 0.62e-7,
// 0.68e-7, 0.73e-7 here and there; halves 0.44e-7, 0.57e-7, 0.76e-7 against 0.44e-7, 0.52e-7, 0.59e-7, row kernels 0.55e-7, 0.62e-7, 0.67e-7).
// (Two heads of fp32, width 128: 297 us along a chain, 306 with two instructions a sum, 310 with one.)
template <typename T, int D>
__device__ __forceinline__ f32x4 mma_rows(const TileRow<T, D>& a, const TileRow<T, D>& b)
{
    constexpr int N = TileRow<T, D>::kChunks;
    f32x4 sum[N];
    if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a.c[i]), __builtin_bit_cast(f16x8, b.c[i]), kNothing, 0, 0, 0);
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            u32x4 c = a.c[i];
            asm volatile("" : "+v"(c)); // (the products of a chunk at a time: all of them at once cost up to 128 registers)
            f32x4 x[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(c[j]), __uint_as_float(b.c[i][j]), kNothing, 0, 0, 0);
            sum[i] = (x[0] + x[1]) + (x[2] + x[3]);
            asm volatile("" : "+v"(sum[i]));
        }
    }
#pragma unroll
    for (int h = 1; h < N; h *= 2)
#pragma unroll
        for (int i = 0; i < N; i += 2 * h) sum[i] += sum[i + h];
    return sum[0];
}

// The dense rows of a step on their way through LDS to operand A: loaded in order (every load 1024 consecutive
// bytes), stored, and read back along or across their elements.  Where 16 bytes are put spreads the
// 16 lanes that LDS serves together (lanes 0-3, 12-15, 20-27 and their like) over all of its banks:
//   kAlong: chunk c of row r at position c ^ f(r) of the row (16 rows are read at one c);
//   kAcross (TileCols, 32-bit sums): the rows of lanes 16 apart, four apart in r, in different parts of 256 bytes;
//   kTransposed (TileCols, halves): 32 bytes each of eight rows are read together, from eight parts of 256 bytes.
enum TileRead { kAlong, kAcross, kTransposed };
template <typename T>
constexpr TileRead tile_columns() // how operand A of the weighted sums is read
{
    return sizeof(T) == 2 ? kTransposed : kAcross;
}
template <typename T, int D, TileRead READ, int ROWS = 16 * tile_blocks<T>()>
struct TileStage {
    static constexpr int kPerRow = D * (int)sizeof(T) / 16; // 16-byte chunks of a row
    static constexpr int kLoads = ROWS * kPerRow / kWave;
    static_assert(ROWS * kPerRow % kWave == 0, "whole loads");
    static constexpr int kBytes = ROWS * kPerRow * 16;
    u32x4 x[kLoads];
    static __device__ __forceinline__ int place(int row, int c)
    {
        if constexpr (READ == kAlong) {
            const int f = kPerRow == 4 ? (-(row >> 2)) & 3 : row & (kPerRow < 16 ? kPerRow - 1 : 15);
            return row * kPerRow + (c ^ f);
        } else if constexpr (READ == kTransposed) {
            constexpr int kRows = kPerRow < 16 ? 16 / kPerRow : 1, kPairs = kPerRow < 16 ? kPerRow / 2 : 8; // (rows in 256 bytes; what f goes up to)
            return row * kPerRow + (c ^ 2 * (row / kRows & (kPairs - 1)));
        } else {
            constexpr int kParts = kPerRow < 16 ? 16 / kPerRow : 1; // rows in 256 bytes
            return (row ^ ((row >> 2) & (kParts - 1))) * kPerRow + c;
        }
    }
    // the rows from `first` on; rows past `last` (counted from there) repeat it
    __device__ __forceinline__ void load(const T* first, int last, bool inside, int lane)
    {
        if (inside) {
#pragma unroll
            for (int i = 0; i < kLoads; ++i) x[i] = reinterpret_cast<const u32x4*>(first)[i * kWave + lane];
        } else {
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                const int at = i * kWave + lane;
                x[i] = reinterpret_cast<const u32x4*>(first)[min(at / kPerRow, last) * kPerRow + at % kPerRow];
            }
        }
    }
    __device__ __forceinline__ void store(u32x4* lds, int lane) const
    {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) lds[place((i * kWave + lane) / kPerRow, (i * kWave + lane) % kPerRow)] = x[i];
    }
    // rows 16 t .. 16 t + 15 as operand A along their elements
    static __device__ __forceinline__ void read(const u32x4* lds, int t, int lane, TileRow<T, D>& row)
    {
#pragma unroll
        for (int i = 0; i < TileRow<T, D>::kChunks; ++i) row.c[i] = lds[place(16 * t + lane % 16, 4 * i + lane / 16)];
    }
    // this lane's D / 16 elements (from (D / 16) n) of row r
    static __device__ __forceinline__ const T* across(const u32x4* lds, int r, int n)
    {
        constexpr int kElems = 16 / (int)sizeof(T), NB = D / 16;
        return reinterpret_cast<const T*>(lds + place(r, NB * n / kElems)) + NB * n % kElems;
    }
    // halves, transposed: element 16 nb + lane % 16 of the rows 16 t + 4 (lane / 16) .. + 3.  (ds_read_b64_tr_b16: of every 16
    // lanes lane 4 r + p names four halves; lane m gets the m-th of the 16 that lanes 4 r .. 4 r + 3 name, for r = 0 .. 3.)
    static __device__ __forceinline__ uint2 transposed(const u32x4* lds, int t, int nb, int lane)
    {
        static_assert(READ == kTransposed && sizeof(T) == 2, "16-bit elements placed for it");
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        const int row = 16 * t + lane / 16 * 4 + lane % 16 / 4, part = lane % 4;
        const T* at = reinterpret_cast<const T*>(lds + place(row, 2 * nb + part / 2)) + part % 2 * 4;
        return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(at)));
    }
};

// One number per (row of the tile, column) of a step, between the layout that memory wants
// (lane 4 r + part: row r, 4 consecutive columns from 4 part on, in each 16-column block) and
// the scores' (lane (n, gq)), through LDS.
template <typename T>
struct TileSquare {
    static constexpr int kFloats = tile_blocks<T>() * kTileRows * 16;
    static __device__ __forceinline__ int place(int t, int row, int part) { return (t * kTileRows + row) * 4 + (part ^ ((-(row >> 2)) & 3)); }
    static __device__ __forceinline__ f32x4& in_order(f32x4* lds, int t, int lane) { return lds[place(t, lane / 4, lane % 4)]; }
    static __device__ __forceinline__ f32x4& as_scores(f32x4* lds, int t, int lane) { return lds[place(t, lane % 16, lane / 16)]; }
};

// ---- weights: operand B of the weighted sums -------------------------------------------------
// fp16 dense operands: a weight is the sum of two halves, each rounded to nearest.  Weights are kept below 2^15 by a power of
// two; from 2^-2 on the sum is within 2^-23 of the weight (a 32-bit number: 2^-24), below that within 2^-25 of it in all.
template <typename T>
struct TileWeights;
template <>
struct TileWeights<__half> {
    static constexpr float kScale = 0x1p15f; // probabilities are taken times that
    f16x8 hi, lo;
    // the weights p times a power of two (the small part by v_fma_mix: a product, a difference and a rounding in one)
    __device__ __forceinline__ void set(const float (&p)[8], float scale)
    {
        u32x4 pairs;
#pragma unroll
        for (int j = 0; j < 8; j += 2) pairs[j / 2] = __builtin_bit_cast(unsigned, f16x2{(_Float16)(p[j] * scale), (_Float16)(p[j + 1] * scale)});
        asm volatile("" : "+v"(pairs)); // (rounded once, in pairs: the compiler would round each again for the difference)
        hi = __builtin_bit_cast(f16x8, pairs);
#pragma unroll
        for (int j = 0; j < 8; ++j) lo[j] = (_Float16)fmaf(p[j], scale, -(float)hi[j]);
    }
};
template <>
struct TileWeights<float> {
    static constexpr float kScale = 1.f;
    float p[4];
    __device__ __forceinline__ void set(const float (&w)[4], float)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = w[j];
    }
};

// ---- columns: a lane's 4 or 8 dense rows across their elements, operand A of the weighted sums ----
// (accumulate: halves along one chain of products per wave, the small parts of a step's weights before the large ones; fp32 a
// chain per step and the steps' sums added, as one chain over a wave's columns - 128 roundings of a growing sum where the row kernels
// have 72 and a tree - had 1.3 to 1.6 times their error)
template <typename T, int D>
struct TileCols;
template <int D>
struct TileCols<__half, D> {
    static constexpr int kBlocks = D / 16;
    using Stage = TileStage<__half, D, kTransposed>;
    uint2 w[kBlocks][2];
    __device__ __forceinline__ void load(const u32x4* lds, int lane)
    {
#pragma unroll
        for (int nb = 0; nb < kBlocks; ++nb)
#pragma unroll
            for (int t = 0; t < 2; ++t) w[nb][t] = Stage::transposed(lds, t, nb, lane);
    }
    __device__ __forceinline__ void accumulate(const TileWeights<__half>& p, f32x4 (&acc)[kBlocks]) const
    {
#pragma unroll
        for (int nb = 0; nb < kBlocks; ++nb) {
            const f16x8 a = __builtin_bit_cast(f16x8, make_uint4(w[nb][0].x, w[nb][0].y, w[nb][1].x, w[nb][1].y));
            acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, p.lo, acc[nb], 0, 0, 0);
            acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, p.hi, acc[nb], 0, 0, 0);
        }
    }
    // the c'th four consecutive elements of this lane's sums, and where they are in the row
    static __device__ __forceinline__ f32x4 sums(const f32x4 (&acc)[kBlocks], int c) { return acc[c]; }
    static __device__ __forceinline__ int at(int c, int gq) { return 16 * c + 4 * gq; }
};
template <int D>
struct TileCols<float, D> {
    static constexpr int kBlocks = D / 16;
    using Stage = TileStage<float, D, kAcross>;
    float x[4][kBlocks];
    __device__ __forceinline__ void load(const u32x4* lds, int lane)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j) load(j, Stage::across(lds, lane / 16 * 4 + j, lane % 16));
    }
    __device__ __forceinline__ void load(int j, const float* at)
    {
        if constexpr (kBlocks == 2) {
            const float2 v = *reinterpret_cast<const float2*>(at);
            x[j][0] = v.x, x[j][1] = v.y;
        } else {
#pragma unroll
            for (int b = 0; b < kBlocks; b += 4) {
                const float4 v = *reinterpret_cast<const float4*>(at + b);
                x[j][b] = v.x, x[j][b + 1] = v.y, x[j][b + 2] = v.z, x[j][b + 3] = v.w;
            }
        }
    }
    __device__ __forceinline__ void load(int j, const __half* at) // (widened)
    {
#pragma unroll
        for (int b = 0; b < kBlocks; b += 2) {
            const float2 v = __half22float2(*reinterpret_cast<const __half2*>(at + b));
            x[j][b] = v.x, x[j][b + 1] = v.y;
        }
    }
    __device__ __forceinline__ void accumulate(const TileWeights<float>& p, f32x4 (&acc)[kBlocks]) const
    {
        constexpr int kAtOnce = kBlocks < 4 ? kBlocks : 4;
#pragma unroll
        for (int b = 0; b < kBlocks; b += kAtOnce) {
            f32x4 sum[kAtOnce];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < kAtOnce; ++i) sum[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j][b + i], p.p[j], j == 0 ? kNothing : sum[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < kAtOnce; ++i) acc[b + i] += sum[i];
        }
    }
    static __device__ __forceinline__ f32x4 sums(const f32x4 (&acc)[kBlocks], int c)
    {
        f32x4 e;
#pragma unroll
        for (int x = 0; x < 4; ++x) e[x] = acc[(4 * c + x) % kBlocks][(4 * c + x) / kBlocks];
        return e;
    }
    static __device__ __forceinline__ int at(int c, int gq) { return D / 4 * gq + 4 * c; }
};

template <int NB>
__device__ __forceinline__ bool all_finite(const f32x4 (&acc)[NB])
{
    float s = 0.f; // (a sum of x * 0 is zero, or NaN as soon as one x is not finite)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) s = fmaf(acc[b][i], 0.f, s);
    return s == 0.f;
}

// One lane's row of a tile: its nonzeros, and the run of consecutive columns among them.
struct TileLane {
    int row, s, e;    // slots [s, e)
    int a, len, pos;  // columns [a, a + len) from slot s + pos on
    __device__ __forceinline__ int base() const { return s + pos - a; } // slot of column c of the run: base() + c
    __device__ __forceinline__ int4 packed() const { return make_int4(s, e - s, pos, len); }
};
__device__ __forceinline__ TileLane tile_lane(int row, const int* __restrict__ row_ptr, const int* __restrict__ runs)
{
    TileLane t;
    t.row = row;
    t.s = row_ptr[row], t.e = row_ptr[row + 1];
    t.a = runs[3 * row], t.len = runs[3 * row + 1], t.pos = runs[3 * row + 2];
    return t;
}

// ---- the nonzeros outside the runs -------------------------------------------------------------
// A wave has four rows of the tile and 16 lanes for the nonzeros of each (kOutsideSteps of them per lane at a time): the rows'
// dependent steps - columns, dense rows, reductions, the softmax - then go on side by side instead of one row after
// the other, and each lane group's sums belong to one row (width 128 in fp32: to two, kRows).
constexpr int kOutsideRows = kTileRows / kWavesPerWg, kOutsideSteps = 4;
static_assert(kOutsideRows * 16 == kWave, "16 lanes per row");
template <typename T, int D>
struct TileOutside {
    static constexpr int kVec = 16 / (int)sizeof(T), kLpr = D / kVec, kRows = kLpr > 16 ? kLpr / 16 : 1; // (rows of a lane group)
    static constexpr int kQuads = kLpr / 4 / kRows;                                                       // quads of a row per lane group and step
    int mine, first, split, jump, cnt, most; // this lane's row (of the tile) and its nonzeros; the most that one of the four rows has
    int cnt_of[kRows];                       // a row of this lane group has work in the step from nonzero n on while n < cnt_of
    int group;
    // (rows: what tile_lane says of every row of the tile, TileLane::packed)
    __device__ __forceinline__ TileOutside(const int4* rows, int wave, int lane, bool whole) : group(lane / kLpr)
    {
        mine = kOutsideRows * wave + lane / 16;
        const int4 r = rows[mine];
        first = r.x, split = r.z, jump = whole ? 0 : r.w;
        cnt = r.y - jump;
        most = 0;
#pragma unroll
        for (int i = 0; i < kOutsideRows; ++i) most = max(most, __builtin_amdgcn_readlane(cnt, 16 * i));
#pragma unroll
        for (int i = 0; i < kRows; ++i) cnt_of[i] = kRows == 1 ? cnt - group * kLpr % 16 : __shfl(cnt, group * kLpr + 16 * i, kWave);
    }
    // row i of this lane group (of the tile)
    __device__ __forceinline__ int row(int i) const { return kRows == 1 ? mine : (mine & ~(kRows - 1)) + i; }
    // where nonzero `at` of this lane's row is (past the end: its last one)
    __device__ __forceinline__ int slot(int at) const
    {
        at = min(at, cnt - 1);
        return first + at + (at >= split ? jump : 0);
    }
    // acc += the kQuads quads of weights from `from` on times their dense rows (a sum of their own first)
    static __device__ __forceinline__ void add(const char* dense, unsigned lane_at, const unsigned* row_at, const float* weight, int from, float (&acc)[kVec])
    {
        u32x4 raw[kQuads][4];
#pragma unroll
        for (int u = 0; u < kQuads; ++u) {
            const u32x4 o = *reinterpret_cast<const u32x4*>(row_at + from + 4 * u);
#pragma unroll
            for (int j = 0; j < 4; ++j) raw[u][j] = *reinterpret_cast<const u32x4*>(dense + (o[j] + lane_at));
        }
        float sum[kVec];
#pragma unroll
        for (int u = 0; u < kQuads; ++u) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(weight + from + 4 * u);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float b[kVec];
                DenseVec<T>::unpack(make_uint4(raw[u][j][0], raw[u][j][1], raw[u][j][2], raw[u][j][3]), b);
#pragma unroll
                for (int x = 0; x < kVec; ++x) sum[x] = u == 0 && j == 0 ? w[j] * b[x] : fmaf(w[j], b[x], sum[x]);
            }
        }
#pragma unroll
        for (int x = 0; x < kVec; ++x) acc[x] += sum[x];
    }
    // the four rows' sums to LDS, `stride` floats apart
    __device__ __forceinline__ void store(float (&acc)[kRows][kVec], float* to, int stride, int lane) const
    {
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            if constexpr (kLpr < 16) { // (several lane groups have a row)
#pragma unroll
                for (int x = 0; x < kVec; ++x) acc[i][x] = butterfly_sum<kLpr, 16>(acc[i][x]);
            }
            if (kLpr >= 16 || group % (16 / (kLpr < 16 ? kLpr : 16)) == 0) {
#pragma unroll
                for (int x = 0; x < kVec; x += 4)
                    *reinterpret_cast<f32x4*>(to + row(i) % kOutsideRows * stride + lane % kLpr * kVec + x) = f32x4{acc[i][x], acc[i][x + 1], acc[i][x + 2], acc[i][x + 3]};
            }
        }
    }
};

} // namespace rode
