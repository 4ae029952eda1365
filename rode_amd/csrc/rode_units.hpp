// Inner loops shared by the SDDMM, SpMM and fused attention kernels: the dot products of
// one 32-slot unit (SDDMM), the gather-accumulate over staged slot quads (SpMM) and a step of the
// running softmax (attention).
#pragma once
#include "rode_device.hpp"

namespace rode {

// ---- SDDMM ------------------------------------------------------------------
// KT = width of the lane tile (32, 64 or 128 elements): LPR = KT / VEC lanes read KT
// consecutive elements of a dense row per load instruction.  A row of K elements is
// covered by NS such slabs (KT * NS >= K); EDGE (kPartial, kPartialApart) says that the last slab is partial, in
// which case the lanes past K contribute zero.
constexpr int kPartial = 1;
constexpr int kPartialApart = 2; // ... and the loads of the slots come one by one (lane_dot)
template <typename T, int KT>
struct SddmmShape {
    static constexpr int kVec = DenseVec<T>::kElems;
    static constexpr int kRegs = DotVec<T>::kRegs; // registers of a lane's part of the lhs row
    using Reg = typename DotVec<T>::Reg;
    static constexpr int kLpr = KT / kVec;     // lanes that cover one slab of a dense row
    static constexpr int kQuads = kLpr / 4;    // slot quads per lane group per unit
    static_assert(KT % kVec == 0 && kLpr >= 4 && kLpr <= 32 && (kLpr & (kLpr - 1)) == 0,
                  "unsupported tile width for this dense type");
};

// <lhs row, rhs row> restricted to this lane's elements.  A lane past K reads the row's last elements and drops what it makes of them: loads
// under a condition are sent one by one, each waited for (us, SDDMM of width 96, condition -> none: 29 K rows of 12 28.0 -> 19.4, 100 K of 20 154
// -> 104, power law 200 K 428 -> 250; halves 88 -> 67; width 48 88 -> 66; 4000 rows of 40 8.3 either way, x 100 8.2 -> 8.4, with the row's first
// elements 8.7).  kPartialApart keeps the condition, for the calls that are faster with it (loads_apart, rode_sddmm.hip).
template <typename T, int KT, int NS, int EDGE>
__device__ __forceinline__ float lane_dot(const typename DotVec<T>::Reg (&a)[NS][DotVec<T>::kRegs],
                                          const T* __restrict__ row_lane, int k, int lane_elem)
{
    float d = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const bool ok = !EDGE || lane_elem + s * KT < k;
        if constexpr (EDGE == kPartialApart) {
            if (ok) d = DotVec<T>::dot(a[s], row_lane + s * KT, d);
            continue;
        }
        const float more = DotVec<T>::dot(a[s], row_lane + (ok ? s * KT : k - SddmmShape<T, KT>::kVec - lane_elem), d);
        d = ok ? more : d;
    }
    return d;
}

// The sums over the LPR lanes of a dense row of four slots' partial products: a
// transpose-reduce, after which lane (ls & 3) == j holds slot j of the quad.
template <int LPR>
__device__ __forceinline__ float sddmm_quad_reduce(const float (&p)[4], int ls)
{
    const bool hi2 = ls & 2, hi1 = ls & 1;
    const float k0 = hi2 ? p[2] : p[0], s0 = hi2 ? p[0] : p[2];
    const float k1 = hi2 ? p[3] : p[1], s1 = hi2 ? p[1] : p[3];
    const float q0 = k0 + lane_xor2(s0);
    const float q1 = k1 + lane_xor2(s1);
    const float r = (hi1 ? q1 : q0) + lane_xor1(hi1 ? q0 : q1);
    return butterfly_sum<4, LPR>(r);
}

// Dot products of the 32-slot units of one step, the slots' columns already in lds_cols
// (lds_cols[e] = column of lane e's slot).  Returns the dot product for this lane's slot.
template <typename T, int KT, int NS, int EDGE>
__device__ __forceinline__ float sddmm_unit_staged(const T* __restrict__ rhs_lane,
                                                   const typename DotVec<T>::Reg (&a)[NS][DotVec<T>::kRegs], int k,
                                                   const int* lds_cols, int lane)
{
    using S = SddmmShape<T, KT>;
    constexpr int LPR = S::kLpr;
    const int ls = lane % LPR;                    // lane inside its group
    const int group_first = (lane & 31) - ls;     // first slot (within the half) of this group
    const int* group_cols = lds_cols + (lane & 32) + group_first;
    float result = 0.f;

#pragma unroll
    for (int q = 0; q < S::kQuads; ++q) {
        const int4 c4 = *reinterpret_cast<const int4*>(group_cols + 4 * q);
        const int c[4] = {c4.x, c4.y, c4.z, c4.w};
        float p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            p[j] = lane_dot<T, KT, NS, EDGE>(a, rhs_lane + (size_t)c[j] * k, k, ls * S::kVec);
        const float r = sddmm_quad_reduce<LPR>(p, ls);
        if ((ls >> 2) == q) result = r;
    }
    return result;
}

// Dot products of one 32-slot unit of a block segment.  `my_col` is the column of this
// lane's slot.  Returns the dot product for this lane's slot.
template <typename T, int KT, int NS, int EDGE>
__device__ __forceinline__ float sddmm_unit(const T* __restrict__ rhs_lane,
                                            const typename DotVec<T>::Reg (&a)[NS][DotVec<T>::kRegs], int my_col, int k,
                                            int* lds_cols, int lane)
{
    lds_cols[lane] = my_col;
    wave_lds_sync();
    return sddmm_unit_staged<T, KT, NS, EDGE>(rhs_lane, a, k, lds_cols, lane);
}

// ONCE: the row is used by this work item only (a residue row): loaded with the non-temporal
// hint, so that the stream of lhs rows does not displace gathered rhs rows (config 4: residue
// kernel 1.375 -> 1.334 ms at K=128, 0.656 -> 0.626 at K=64; for the group kernels, which
// read their lhs rows twice, the hint costs 8 %).
template <typename T, int KT, int NS, int EDGE, bool ONCE = false>
__device__ __forceinline__ void load_lhs_slice(const T* __restrict__ lhs, int row, int k, int lane,
                                               typename DotVec<T>::Reg (&a)[NS][DotVec<T>::kRegs])
{
    using S = SddmmShape<T, KT>;
    const int e0 = (lane % S::kLpr) * S::kVec;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        DotVec<T>::zero(a[s]);
        if (!EDGE || e0 + s * KT < k) {
            if constexpr (ONCE)
                DotVec<T>::load_once(lhs + (size_t)row * k + e0 + s * KT, a[s]);
            else
                DotVec<T>::load(lhs + (size_t)row * k + e0 + s * KT, a[s]);
        }
    }
}

// ---- SpMM -------------------------------------------------------------------
template <typename T, int TN>
struct SpmmShape {
    using Acc = typename DenseVec<T>::Acc;          // type of values, accumulators and C
    static constexpr int kVec = DenseVec<T>::kElems;
    static constexpr int kLpr = TN / kVec;          // lanes that cover one B-row tile
    static constexpr int kGroupsWave = kWave / kLpr; // lane groups per wave
    static_assert(TN % kVec == 0 && kLpr >= 4 && kLpr <= 32 && (kLpr & (kLpr - 1)) == 0,
                  "unsupported tile width for this dense type");
};

__device__ __forceinline__ void load_quad(const float* p, float (&v)[4])
{
    const float4 t = *reinterpret_cast<const float4*>(p);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}
__device__ __forceinline__ void load_quad(const double* p, double (&v)[4])
{
    const double2 t0 = *reinterpret_cast<const double2*>(p), t1 = *reinterpret_cast<const double2*>(p + 2);
    v[0] = t0.x; v[1] = t0.y; v[2] = t1.x; v[3] = t1.y;
}

// acc += sum over the slot quads {first_quad, first_quad + stride, ...} < nquads of
// value * B[col, tile].  QUADS_MAX bounds the trip count at compile time.
// EIGHTS: every quad has a sum of its own, and two of them are added before they are added to acc: an eighth of the additions in one chain (for
// tiles that a narrower one would do, with as many times fewer lane groups).
template <typename T, int TN, int QUADS_MAX, bool FULL, bool EIGHTS = false>
__device__ __forceinline__ void spmm_gather(const T* __restrict__ b_lane, size_t ldb,
                                            typename DenseVec<T>::Acc (&acc)[SpmmShape<T, TN>::kVec],
                                            const int* lds_col, const typename DenseVec<T>::Acc* lds_val,
                                            int first_quad, int stride, int nquads)
{
    using A = typename DenseVec<T>::Acc;
    constexpr int VEC = SpmmShape<T, TN>::kVec;
    static_assert(!EIGHTS || QUADS_MAX % 2 == 0, "two quads at a time");
    A two[VEC];
#pragma unroll
    for (int i = 0; i < QUADS_MAX; ++i) {
        const int q = first_quad + i * stride;
        if (FULL || q < nquads) {
            const int4 c4 = *reinterpret_cast<const int4*>(lds_col + 4 * q);
            const int c[4] = {c4.x, c4.y, c4.z, c4.w};
            A v[4];
            load_quad(lds_val + 4 * q, v);
            A b[4][VEC];
#pragma unroll
            for (int j = 0; j < 4; ++j) DenseVec<T>::load(b_lane + (size_t)c[j] * ldb, b[j]);
            if constexpr (EIGHTS) {
#pragma unroll
                for (int x = 0; x < VEC; ++x) {
                    A sum = A(0);
#pragma unroll
                    for (int j = 0; j < 4; ++j) sum = fma(v[j], b[j][x], sum);
                    two[x] = i % 2 ? two[x] + sum : sum;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int x = 0; x < VEC; ++x) acc[x] = fma(v[j], b[j][x], acc[x]);
            }
        }
        if constexpr (EIGHTS) {
            const int first = q - (i % 2) * stride; // (the pair's first quad)
            if (i % 2 == 1 && (FULL || first < nquads)) {
#pragma unroll
                for (int x = 0; x < VEC; ++x) acc[x] += two[x];
            }
            // (32-bit operands: the loads of half of the quads at a time.  Of all of them together 131 registers, three waves per SIMD: 4000 rows of
            // 56 x 96 7.2 -> 8.8 us)
            if (FULL && VEC == 4 && i + 1 == QUADS_MAX / 2) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The same sum over the quads 0 .. nquads - 1, two quads per step: the loads of both are
// issued before either is used (eight dense rows in flight per lane instead of four), and a
// quad that does not exist loads nothing and adds zeros.  For work items of a few quads
// whose kernels are bound by memory latency (residue rows).
template <typename T, int TN, int QUADS_MAX>
__device__ __forceinline__ void spmm_gather_pairs(const T* __restrict__ b_lane, size_t ldb,
                                                  typename DenseVec<T>::Acc (&acc)[SpmmShape<T, TN>::kVec],
                                                  const int* lds_col, const typename DenseVec<T>::Acc* lds_val, int nquads)
{
    using A = typename DenseVec<T>::Acc;
    constexpr int VEC = SpmmShape<T, TN>::kVec;
    static_assert(QUADS_MAX % 2 == 0, "two quads per step");
#pragma unroll
    for (int q = 0; q < QUADS_MAX; q += 2) {
        if (q < nquads) {
            A v[2][4], b[2][4][VEC];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[h][j] = A(0);
#pragma unroll
                    for (int x = 0; x < VEC; ++x) b[h][j][x] = A(0);
                }
                if (q + h < nquads) {
                    const int4 c4 = *reinterpret_cast<const int4*>(lds_col + 4 * (q + h));
                    const int c[4] = {c4.x, c4.y, c4.z, c4.w};
                    load_quad(lds_val + 4 * (q + h), v[h]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) DenseVec<T>::load(b_lane + (size_t)c[j] * ldb, b[h][j]);
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int x = 0; x < VEC; ++x) acc[x] = fma(v[h][j], b[h][j][x], acc[x]);
        }
    }
}

// A row of C that is written once and not read again by the kernel that writes it: stored
// with the non-temporal hint, so that it does not push the gathered rows of B out of the
// caches on its way (config 4, K=128: residue kernel 1.19 -> 1.09 ms; the same hint on the
// loads of B, on SDDMM's loads of rhs or on its stores of `out` made those kernels slower).
template <int VEC>
__device__ __forceinline__ void store_row(float* dst, const float (&acc)[VEC])
{
    typedef float Quad __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int x = 0; x < VEC; x += 4) {
        const Quad v = {acc[x], acc[x + 1], acc[x + 2], acc[x + 3]};
        __builtin_nontemporal_store(v, reinterpret_cast<Quad*>(dst + x));
    }
}

template <int VEC>
__device__ __forceinline__ void store_row(double* dst, const double (&acc)[VEC])
{
    typedef double Pair __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int x = 0; x < VEC; x += 2) {
        const Pair v = {acc[x], acc[x + 1]};
        __builtin_nontemporal_store(v, reinterpret_cast<Pair*>(dst + x));
    }
}

// ---- attention ----------------------------------------------------------------
// What a kernel leaves behind for the gradient.
enum Keep : int {
    kKeepNothing = 0,
    kKeepProbs = 1,  // probs[idx] = the probability
    kKeepScores = 2, // probs[idx] = the scaled score, stats[row] = (row maximum, 1 / row sum)
};

// One step of the running softmax of a row: the scores of up to 64 slots (sc, -inf for a
// lane without a slot) move the maximum; the row's sum and accumulated output are rescaled.
// Returns this lane's probability relative to the new maximum.
template <int VEC>
__device__ __forceinline__ float softmax_step(float sc, bool live, float& m_run, float& l_lane, float (&acc)[VEC])
{
    const float m_new = fmaxf(m_run, butterfly_max<1, kWave>(sc));
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float corr = __expf(m_run - m_safe);
    const float p = live ? __expf(sc - m_safe) : 0.f;
    l_lane = fmaf(l_lane, corr, p);
    if (m_run != -INFINITY) { // (nothing to rescale before the first step)
#pragma unroll
        for (int x = 0; x < VEC; ++x) acc[x] *= corr;
    }
    m_run = m_new;
    return p;
}

// ---- attention, column pass of the gradient ----------------------------------------
// Lane layout of the column pass for every operand type: D / 4 lanes per dense row, four
// elements each (g is fp32 whatever q is, and both feed accumulators of the same shape).
__device__ __forceinline__ void load4(const float* p, float (&out)[4])
{
    const float4 t = *reinterpret_cast<const float4*>(p);
    out[0] = t.x; out[1] = t.y; out[2] = t.z; out[3] = t.w;
}
__device__ __forceinline__ void load4(const __half* p, float (&out)[4])
{
    const uint2 raw = *reinterpret_cast<const uint2*>(p);
    const float2 lo = __half22float2(*reinterpret_cast<const __half2*>(&raw.x));
    const float2 hi = __half22float2(*reinterpret_cast<const __half2*>(&raw.y));
    out[0] = lo.x; out[1] = lo.y; out[2] = hi.x; out[3] = hi.y;
}

// dv += p * g[row], dk += dz * q[row] over the slot quads {first_quad, first_quad + stride, ...}
// < nquads of a staged step (rows, p and dz of the slots in LDS).
template <typename T, int D, int QUADS_MAX, bool FULL>
__device__ __forceinline__ void cols_gather(const float* __restrict__ g_lane, const T* __restrict__ q_lane,
                                            float (&acc_v)[4], float (&acc_k)[4], const int* lds_row,
                                            const float* lds_p, const float* lds_z, int first_quad, int stride, int nquads)
{
#pragma unroll
    for (int i = 0; i < QUADS_MAX; ++i) {
        const int qd = first_quad + i * stride;
        if (FULL || qd < nquads) {
            const int4 r4 = *reinterpret_cast<const int4*>(lds_row + 4 * qd);
            const int r[4] = {r4.x, r4.y, r4.z, r4.w};
            float pv[4], zv[4], bg[4][4], bq[4][4];
            load_quad(lds_p + 4 * qd, pv);
            load_quad(lds_z + 4 * qd, zv);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                load4(g_lane + (size_t)r[t] * D, bg[t]);
                load4(q_lane + (size_t)r[t] * D, bq[t]);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    acc_v[x] = fmaf(pv[t], bg[t][x], acc_v[x]);
                    acc_k[x] = fmaf(zv[t], bq[t][x], acc_k[x]);
                }
        }
    }
}

} // namespace rode
