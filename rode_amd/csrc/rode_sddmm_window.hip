// SDDMM for the chunks of the residue list whose dense rows cluster in a window (banded
// matrices; see rode_window.hpp for the shape of the kernel and rode_plan.hip for how
// the chunks are chosen).  Same rows and slots as sddmm_residue_kernel in rode_sddmm.hip
// (reference: RoDe_SDDMM/RoDeSddmm.cu:206-494); what differs is where the rhs rows come
// from, and that a lane keeps, for every slot of its row, the partial dot product over its own 16
// bytes of all column tiles; the 8 lanes of a row are summed once, after the last tile, with a
// transpose-reduce (DPP) that leaves position 8i + l in lane l.  Every tile has a sum of its own: with one
// chain over the tiles the errors were 5 % (two tiles) and 17 % (four) larger (2-norm against 64 bits: fp32 of width 64 7.6e-8 -> 7.2e-8, of
// 128 9.1e-8 -> 7.8e-8, 128 halves 7.6e-8 -> 7.2e-8); 1 M rows of 27: 244 -> 245, 383 -> 386, 263 -> 278 us.
#include "rode_window.hpp"
#include "rode_internal.hpp"

namespace rode {

namespace {

// Sum over the 8 lanes of a group of 8 per-lane values; lane l returns the total of p[l].
__device__ __forceinline__ float transpose_reduce8(const float (&p)[8], int ls)
{
    const bool b2 = ls & 4, b1 = ls & 2, b0 = ls & 1;
    float r4[4], r2[2];
#pragma unroll
    for (int k = 0; k < 4; ++k) r4[k] = (b2 ? p[k + 4] : p[k]) + lane_xor4(b2 ? p[k] : p[k + 4]);
#pragma unroll
    for (int k = 0; k < 2; ++k) r2[k] = (b1 ? r4[k + 2] : r4[k]) + lane_xor2(b1 ? r4[k] : r4[k + 2]);
    return (b0 ? r2[1] : r2[0]) + lane_xor1(b0 ? r2[0] : r2[1]);
}

template <typename T, bool EDGE>
__global__ void __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
sddmm_residue_window_kernel(int m2, int k, const int* __restrict__ col, const float* __restrict__ val,
                            const T* __restrict__ lhs, const T* __restrict__ rhs, float* __restrict__ out,
                            const PlannedChunk* __restrict__ rows)
{
    constexpr int VEC = DenseVec<T>::kElems;
    constexpr int TW = kResLanes * VEC; // elements of a dense row in one tile
    constexpr int QUADS = kBlockItems / 4;
    constexpr int OWN = kBlockItems / kResLanes;
    __shared__ uint4 win[2 * kResWinVecs];
    __shared__ uint4 records[2 * kRecordRoom];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int group = threadIdx.x / kResLanes, ls = threadIdx.x % kResLanes;
    const ChunkWalk walk(m2);
    int chunk = walk.from(rows, walk.at);
    if (chunk >= walk.end) return;
    const int tiles = (k + TW - 1) / TW; // at least two
    const char* win_bytes = reinterpret_cast<const char*>(win);
    const unsigned win_lds = lds_address(win), rec_lds = lds_address(records);

    auto window = [&](int w0, int wn, int tile, int buf) __attribute__((always_inline)) {
        const unsigned at = EDGE && tile * TW + ls * VEC >= k ? 0u : ls * 16u; // (lanes past the last column do not use theirs)
        fetch_window(win_lds + buf * kResWinVecs * 16, rhs + (size_t)w0 * k + tile * TW, (unsigned)k * (unsigned)sizeof(T), wn, at, wave);
    };
    auto lhs_tile = [&](int row, int tile) __attribute__((always_inline)) {
        const int at = tile * TW + ls * VEC;
        return (!EDGE || at < k) && row >= 0 ? *reinterpret_cast<const uint4*>(lhs + (size_t)row * k + at) : make_uint4(0, 0, 0, 0);
    };
    auto record = [&](int rec) __attribute__((always_inline)) -> const PlannedChunk& {
        return *reinterpret_cast<const PlannedChunk*>(records + rec * kRecordRoom);
    };

    int w0 = rows[chunk].w0, wn = rows[chunk].wn;
    fetch_record(rec_lds, rows + chunk, wave);
    window(w0, wn, 0, 0);
    copies_done();
    __syncthreads();
    uint4 a_next = lhs_tile(record(0).meta[group].row, 0);
    int rec = 0, buf = 0;
    // the dot products of the last chunk, stored during the next one: nobody waits for the stores then
    float result[OWN];
    int result_at[OWN];
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        result[i] = 0.f;
        result_at[i] = -1;
    }

    while (true) {
        const int after = walk.from(rows, chunk + walk.stride);
        const bool last = after >= walk.end;
        const int after_w0 = last ? 0 : rows[after].w0, after_wn = last ? 0 : rows[after].wn;
        ResidueRow rr;
        float v[OWN];
        float acc[kBlockItems]; // this lane's share of every position
#pragma unroll
        for (int i = 0; i < kBlockItems; ++i) acc[i] = 0.f;
        int wave_quads = 0;
        bool wave_all_hit = true;
        for (int tile = 0; tile < tiles; ++tile) {
            copies_done();
            __syncthreads(); // this tile (and the chunk's record) is in LDS, and every wave is done with the one before
            uint4 a_raw = a_next;
            if (tile == 0) {
                decode_planned_row(record(rec), group, 0, rr);
                wave_quads = wave_max_quads((rr.cnt + 3) / 4);
                wave_all_hit = __ballot(rr.missmask != 0) == 0ull;
                if (!last) fetch_record(rec_lds + (rec ^ 1) * kRecordRoom * 16, rows + after, wave);
            }
            asm volatile("" : "+v"(a_raw.x), "+v"(a_raw.y), "+v"(a_raw.z), "+v"(a_raw.w)); // waited for here, before the copies below
            if (tile + 1 < tiles) {
                window(w0, wn, tile + 1, buf ^ 1);
                a_next = lhs_tile(rr.row, tile + 1);
            } else if (!last) {
                window(after_w0, after_wn, 0, buf ^ 1);
                a_next = lhs_tile(record(rec ^ 1).meta[group].row, 0);
            }
            if (tile == 0) {
#pragma unroll
                for (int i = 0; i < OWN; ++i) {
                    if (result_at[i] >= 0) out[result_at[i]] = result[i];
                    const int pos = i * kResLanes + ls;
                    result_at[i] = pos < rr.cnt ? rr.first + planned_slot(record(rec), group, pos) : -1;
                    v[i] = result_at[i] >= 0 ? val[result_at[i]] : 0.f;
                }
            }
            __builtin_amdgcn_sched_barrier(0); // the loads above are issued before the work below, not after it
            const int col_off = tile * TW + ls * VEC;
            const bool col_ok = !EDGE || col_off < k;
            const T* rhs_lane = rhs + (col_ok ? col_off : 0);
            typename DotVec<T>::Reg a[DotVec<T>::kRegs];
            {
                const uint32_t w[4] = {a_raw.x, a_raw.y, a_raw.z, a_raw.w};
                DotVec<T>::load(reinterpret_cast<const T*>(w), a);
            }
            const unsigned base = (unsigned)buf << 16;
            int first_t = rr.first;
            unsigned miss_t = rr.missmask;
            // (opaque: not the tests and addresses of all positions, computed once and held in registers)
            if (!wave_all_hit) asm volatile("" : "+v"(first_t), "+v"(miss_t));
#pragma unroll
            for (int q = 0; q < QUADS; ++q) {
                if (q < wave_quads) { // the same for every lane of the wave
                    uint4 raw[4];
#pragma unroll
                    for (int j = 0; j < 4; j += 2) {
                        unsigned pair = rr.addr[2 * q + j / 2];
                        asm volatile("" : "+v"(pair)); // unpacked here, per tile, not once for all tiles
                        raw[j] = *reinterpret_cast<const uint4*>(win_bytes + window_offset<0>(pair, base));
                        raw[j + 1] = *reinterpret_cast<const uint4*>(win_bytes + window_offset<1>(pair, base));
                    }
                    if (!wave_all_hit) {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if ((miss_t >> (4 * q + j)) & 1u) { // outside the window
                                const int c = col[first_t + planned_slot(record(rec), group, 4 * q + j)];
                                raw[j] = *reinterpret_cast<const uint4*>(rhs_lane + (size_t)c * k);
                            }
                    }
                    if (col_ok) { // (lanes past the last column add nothing)
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[4 * q + j] += DotVec<T>::dot_raw(a, raw[j], 0.f); // (a sum of its own per tile)
                    }
                }
            }
            buf ^= 1;
        }
        // lane l of the group has the positions l, 8 + l, 16 + l, 24 + l
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
            float part8[kResLanes];
#pragma unroll
            for (int j = 0; j < kResLanes; ++j) part8[j] = acc[i * kResLanes + j];
            result[i] = v[i] * transpose_reduce8(part8, ls);
        }
        if (last) break;
        chunk = after;
        w0 = after_w0;
        wn = after_wn;
        rec ^= 1;
    }
#pragma unroll
    for (int i = 0; i < OWN; ++i)
        if (result_at[i] >= 0) out[result_at[i]] = result[i];
}

template <typename T, int TILES>
__global__ void __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
sddmm_ring_kernel(int m2, int k, bool all_windows, const int* __restrict__ plan, const int* __restrict__ col, const float* __restrict__ val, const T* __restrict__ lhs,
                  const T* __restrict__ rhs, float* __restrict__ out, const PlannedChunk* __restrict__ rows)
{
    using R = Ring<TILES>;
    constexpr int VEC = DenseVec<T>::kElems, TW = kResLanes * VEC, QUADS = kBlockItems / 4, OWN = kBlockItems / kResLanes;
    __shared__ uint4 ring[R::kBytes / 16];
    __shared__ uint4 records[3 * kRingRecordVecs];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int group = threadIdx.x / kResLanes, ls = threadIdx.x % kResLanes;
    __shared__ int walk_room[kResThreads / kWave + 2];
    const RingWalk walk(m2, 1, all_windows, plan, walk_room);
    int chunk = walk.from(rows, walk.at);
    if (chunk >= walk.end) return;
    const char* ring_bytes = reinterpret_cast<const char*>(ring);
    const unsigned ring_lds = lds_address(ring), rec_lds = lds_address(records);

    auto fetch_rows = [&](int from, int to) __attribute__((always_inline)) {
        R::fetch(ring_lds, reinterpret_cast<const char*>(rhs), R::kRowBytes, from, to, wave, lane);
    };
    auto fetch_record = [&](int rec, int c) __attribute__((always_inline)) { fetch_ring_record(rec_lds + rec * kRingRecordVecs * 16, rows + c, wave); };
    auto record = [&](int rec) __attribute__((always_inline)) -> const RingRecord& { return *reinterpret_cast<const RingRecord*>(records + rec * kRingRecordVecs); };
    auto lhs_row = [&](const RingRecord& rc, uint4 (&a)[TILES]) __attribute__((always_inline)) {
        const int row = rc.meta[group].row;
#pragma unroll
        for (int t = 0; t < TILES; ++t) a[t] = row >= 0 ? *reinterpret_cast<const uint4*>(lhs + (size_t)row * k + t * TW + ls * VEC) : make_uint4(0, 0, 0, 0);
    };

    int w0 = rows[chunk].w0, low = w0, high = w0 + rows[chunk].wn; // (the ring has rows [low, high))
    int after = walk.from(rows, chunk + 1), rec = 0;
    fetch_rows(low, high);
    fetch_record(0, chunk);
    if (after < walk.end) fetch_record(1, after);
    copies_done();
    __syncthreads();
    uint4 a_next[TILES];
    lhs_row(record(0), a_next);
    // the dot products of the last chunk, stored during the next one: nobody waits for the stores then
    float result[OWN];
    int result_at[OWN];
#pragma unroll
    for (int i = 0; i < OWN; ++i) result[i] = 0.f, result_at[i] = -1;

    while (true) {
        copies_done();
        __syncthreads(); // the chunk's rows and the next one's record are in LDS, and every wave is done with the chunk before
        const RingRecord& mine = record(rec);
        const int4 meta = *reinterpret_cast<const int4*>(&mine.meta[group]);
        const int cnt = meta.x >= 0 ? meta.z & 0xff : 0;
        const unsigned missmask = meta.x >= 0 ? (unsigned)meta.w : 0u;
        unsigned at[kBlockItems / 2];
#pragma unroll
        for (int i = 0; i < kBlockItems / 8; ++i) {
            const uint4 e = reinterpret_cast<const uint4*>(mine.entry[group])[i];
            at[4 * i] = R::units(e.x, w0, ls), at[4 * i + 1] = R::units(e.y, w0, ls), at[4 * i + 2] = R::units(e.z, w0, ls), at[4 * i + 3] = R::units(e.w, w0, ls);
        }
        const int wave_quads = wave_max_quads((cnt + 3) / 4);
        const bool wave_all_hit = __ballot(missmask != 0) == 0ull;
        typename DotVec<T>::Reg a[TILES][DotVec<T>::kRegs];
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            asm volatile("" : "+v"(a_next[t].x), "+v"(a_next[t].y), "+v"(a_next[t].z), "+v"(a_next[t].w)); // waited for here, before the copies below
            const uint32_t w[4] = {a_next[t].x, a_next[t].y, a_next[t].z, a_next[t].w};
            DotVec<T>::load(reinterpret_cast<const T*>(w), a[t]);
        }
        const bool last = after >= walk.end;
        int next_w0 = 0, next_end = 0;
        bool ahead = true;
        const int rec1 = rec == 2 ? 0 : rec + 1, rec2 = rec1 == 2 ? 0 : rec1 + 1;
        int after2 = after;
        if (!last) {
            next_w0 = rows[after].w0, next_end = next_w0 + rows[after].wn;
            const int top = max(high, next_end);
            ahead = next_w0 >= max(low, top - kRingRows) && top - kRingRows <= w0; // do its rows fit beside this chunk's?
            if (ahead) {
                fetch_rows(high, top);
                high = top, low = max(low, top - kRingRows);
            }
            after2 = walk.from(rows, after + 1);
            if (after2 < walk.end) fetch_record(rec2, after2);
            lhs_row(record(rec1), a_next);
        }
        float v[OWN];
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
            if (result_at[i] >= 0) out[result_at[i]] = result[i];
            const int pos = i * kResLanes + ls;
            result_at[i] = pos < cnt ? meta.y + ((mine.entry[group][pos] >> 9) & (kBlockItems - 1)) : -1;
            v[i] = result_at[i] >= 0 ? val[result_at[i]] : 0.f;
        }
        __builtin_amdgcn_sched_barrier(0); // the loads above are issued before the work below, not after it
        float acc[kBlockItems]; // this lane's share of every position
#pragma unroll
        for (int i = 0; i < kBlockItems; ++i) acc[i] = 0.f;
#pragma unroll
        for (int q = 0; q < QUADS; ++q) {
            if (q < wave_quads) { // the same for every lane of the wave
                uint4 raw[TILES][4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const unsigned pair = at[2 * q + j / 2], off = (j % 2 ? pair >> 16 : pair & 0xffffu) << 4;
#pragma unroll
                    for (int t = 0; t < TILES; ++t) raw[t][j] = *reinterpret_cast<const uint4*>(ring_bytes + (off ^ (t * 128u)));
                }
                if (!wave_all_hit) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if ((missmask >> (4 * q + j)) & 1u) { // outside the window
                            const int c = col[meta.y + ((mine.entry[group][4 * q + j] >> 9) & (kBlockItems - 1))];
#pragma unroll
                            for (int t = 0; t < TILES; ++t) raw[t][j] = *reinterpret_cast<const uint4*>(rhs + (size_t)c * k + t * TW + ls * VEC);
                        }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) { // (a sum of its own per tile)
                    acc[4 * q + j] = DotVec<T>::dot_raw(a[0], raw[0][j], 0.f);
#pragma unroll
                    for (int t = 1; t < TILES; ++t) acc[4 * q + j] += DotVec<T>::dot_raw(a[t], raw[t][j], 0.f);
                }
            }
        }
        // lane l of the group has the positions l, 8 + l, 16 + l, 24 + l
#pragma unroll
        for (int i = 0; i < OWN; ++i) {
            float part8[kResLanes];
#pragma unroll
            for (int j = 0; j < kResLanes; ++j) part8[j] = acc[i * kResLanes + j];
            result[i] = v[i] * transpose_reduce8(part8, ls);
        }
        if (last) break;
        if (!ahead) {
            __syncthreads(); // (the rows of a window that lies apart, in the place of this one's)
            fetch_rows(next_w0, next_end);
            low = next_w0, high = next_end;
        }
        w0 = next_w0, rec = rec1, after = after2;
    }
#pragma unroll
    for (int i = 0; i < OWN; ++i)
        if (result_at[i] >= 0) out[result_at[i]] = result[i];
}

} // namespace

// The window kernel over the planned chunks of the residue list, for dense rows that window_takes.
// T = float or __half.
template <typename T>
hipError_t sddmm_window_launch(int m2, int k, const int* col, const float* val, const T* lhs, const T* rhs, float* out,
                               const PlanRef& plan, hipStream_t stream)
{
    if (m2 <= 0) return hipSuccess;
    const size_t row_bytes = (size_t)k * sizeof(T);
    const PlannedChunk* rows = static_cast<const PlannedChunk*>(plan.rows);
    if (plan.rings) {
        if (ring_slices(row_bytes) != 1) return hipErrorInvalidValue;
        const bool all = plan.host_counts != nullptr && plan.host_counts[1] == plan.host_counts[0];
        auto kernel = row_bytes == 128 ? sddmm_ring_kernel<T, 1> : sddmm_ring_kernel<T, 2>;
        kernel<<<kWindowWgs, kResThreads, 0, stream>>>(m2, k, all, plan.dev, col, val, lhs, rhs, out, rows);
        return hipGetLastError();
    }
    if (!window_takes(row_bytes)) return hipErrorInvalidValue;
    auto kernel = ((size_t)k * sizeof(T)) % (kResLanes * 16) != 0 ? sddmm_residue_window_kernel<T, true> : sddmm_residue_window_kernel<T, false>;
    kernel<<<window_grid(m2), kResThreads, 0, stream>>>(m2, k, col, val, lhs, rhs, out, rows);
    return hipGetLastError();
}

template hipError_t sddmm_window_launch<float>(int, int, const int*, const float*, const float*, const float*, float*,
                                               const PlanRef&, hipStream_t);
template hipError_t sddmm_window_launch<__half>(int, int, const int*, const float*, const __half*, const __half*, float*,
                                                const PlanRef&, hipStream_t);

} // namespace rode
