// SpMM for the chunks of the residue list whose dense rows cluster in a window (banded
// matrices; see rode_window.hpp for the shape of the kernel and rode_plan.hip for how
// the chunks are chosen).  Same rows, same slots and the same store/accumulate rule as
// spmm_residue_kernel in rode_spmm.hip (reference: RoDe_SpMM/RoDeSpmm.cu:41-195); what
// differs is where B comes from.
#include "rode_window.hpp"
#include "rode_units.hpp"
#include "rode_internal.hpp"

namespace rode {

namespace {

// 16 bytes of a row of B as numbers of the accumulator's type
template <typename T>
__device__ __forceinline__ void unpack_dense(const uint4& raw, typename DenseVec<T>::Acc (&out)[DenseVec<T>::kElems])
{
    if constexpr (sizeof(T) == 8) {
        out[0] = __hiloint2double((int)raw.y, (int)raw.x);
        out[1] = __hiloint2double((int)raw.w, (int)raw.z);
    } else {
        DenseVec<T>::unpack(raw, out);
    }
}

// lane J of the quad's value
template <int J>
__device__ __forceinline__ float of_quad(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x55 * J, 0xf, 0xf, true));
}
template <int J>
__device__ __forceinline__ double of_quad(double x)
{
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x55 * J, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x55 * J, 0xf, 0xf, true));
}

template <typename T, bool EDGE>
__global__ void __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
spmm_residue_window_kernel(int m2, int n, int owned_slots, const int* __restrict__ col,
                           const typename DenseVec<T>::Acc* __restrict__ val, const T* __restrict__ B,
                           typename DenseVec<T>::Acc* __restrict__ C, const PlannedChunk* __restrict__ rows)
{
    using A = typename DenseVec<T>::Acc;
    constexpr int VEC = DenseVec<T>::kElems;
    constexpr int TW = kResLanes * VEC; // columns of one tile
    constexpr int QUADS = kBlockItems / 4;
    __shared__ uint4 win[2 * kResWinVecs];
    __shared__ uint4 records[2 * kRecordRoom];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int group = threadIdx.x / kResLanes, ls = threadIdx.x % kResLanes;
    const ChunkWalk walk(m2);
    int chunk = walk.from(rows, walk.at);
    if (chunk >= walk.end) return;
    const int tiles = (n + TW - 1) / TW; // at least two
    const char* win_bytes = reinterpret_cast<const char*>(win);
    const unsigned win_lds = lds_address(win), rec_lds = lds_address(records);

    auto window = [&](int w0, int wn, int tile, int buf) __attribute__((always_inline)) {
        const unsigned at = EDGE && tile * TW + ls * VEC >= n ? 0u : ls * 16u; // (lanes past the last column write nothing)
        fetch_window(win_lds + buf * kResWinVecs * 16, B + (size_t)w0 * n + tile * TW, (unsigned)n * (unsigned)sizeof(T), wn, at, wave);
    };
    auto record = [&](int rec) __attribute__((always_inline)) -> const PlannedChunk& {
        return *reinterpret_cast<const PlannedChunk*>(records + rec * kRecordRoom);
    };
    // a row's values lie in the quads of its group: position 4 q + j in lane j
    const int lane_of_quad = ls % 4;
    auto own_values = [&](const PlannedChunk& pc, A (&v)[QUADS]) __attribute__((always_inline)) {
        const int4 meta = *reinterpret_cast<const int4*>(&pc.meta[group]);
#pragma unroll
        for (int q = 0; q < QUADS; ++q) {
            const int pos = 4 * q + lane_of_quad;
            v[q] = meta.x >= 0 && pos < (meta.z & 0xff) ? val[meta.y + planned_slot(pc, group, pos)] : A(0);
        }
    };

    int w0 = rows[chunk].w0, wn = rows[chunk].wn;
    fetch_record(rec_lds, rows + chunk, wave);
    window(w0, wn, 0, 0);
    copies_done();
    __syncthreads();
    A v_next[QUADS];
    own_values(record(0), v_next);
    int rec = 0, buf = 0;
    // a tile's results, written during the next one: nobody waits for the stores then
    A result[VEC];
#pragma unroll
    for (int x = 0; x < VEC; ++x) result[x] = A(0);
    A* result_at = nullptr;
    bool result_adds = false;
    auto write_result = [&]() __attribute__((always_inline)) {
        if (result_at == nullptr) return;
        if (result_adds) {
#pragma unroll
            for (int x = 0; x < VEC; ++x) atomicAdd(result_at + x, result[x]);
        } else {
            store_row<VEC>(result_at, result);
        }
    };

    while (true) {
        const int after = walk.from(rows, chunk + walk.stride);
        const bool last = after >= walk.end;
        const int after_w0 = last ? 0 : rows[after].w0, after_wn = last ? 0 : rows[after].wn;
        ResidueRow rr;
        A v[QUADS];
        int wave_quads = 0;
        bool wave_all_hit = true;
        for (int tile = 0; tile < tiles; ++tile) {
            copies_done();
            __syncthreads(); // this tile (and the chunk's record) is in LDS, and every wave is done with the one before
            if (tile == 0) {
                decode_planned_row(record(rec), group, owned_slots, rr);
                wave_quads = wave_max_quads((rr.cnt + 3) / 4);
                wave_all_hit = __ballot(rr.missmask != 0) == 0ull;
#pragma unroll
                for (int q = 0; q < QUADS; ++q) {
                    v[q] = v_next[q];
                    asm volatile("" : "+v"(v[q])); // waited for here, before the copies below
                }
                if (!last) fetch_record(rec_lds + (rec ^ 1) * kRecordRoom * 16, rows + after, wave);
            }
            if (tile + 1 < tiles) {
                window(w0, wn, tile + 1, buf ^ 1);
            } else if (!last) {
                window(after_w0, after_wn, 0, buf ^ 1);
                own_values(record(rec ^ 1), v_next);
            }
            write_result();
            __builtin_amdgcn_sched_barrier(0); // the loads above are issued before the work below, not after it
            const int col_off = tile * TW + ls * VEC;
            const bool col_ok = !EDGE || col_off < n;
            const T* b_lane = B + (col_ok ? col_off : 0);
            A acc[VEC];
#pragma unroll
            for (int x = 0; x < VEC; ++x) acc[x] = A(0);
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
                            if ((miss_t >> (4 * q + j)) & 1u) { // outside the window: the row of B from memory
                                const int c = col[first_t + planned_slot(record(rec), group, 4 * q + j)];
                                raw[j] = *reinterpret_cast<const uint4*>(b_lane + (size_t)c * n);
                            }
                    }
                    const A v4[4] = {of_quad<0>(v[q]), of_quad<1>(v[q]), of_quad<2>(v[q]), of_quad<3>(v[q])};
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        A b[VEC];
                        unpack_dense<T>(raw[j], b);
#pragma unroll
                        for (int x = 0; x < VEC; ++x) acc[x] = fma(v4[j], b[x], acc[x]);
                    }
                }
            }
            // a listed row without slots of its own (empty, unaligned start) is stored as zeros
            result_adds = rr.accumulate;
            result_at = rr.row >= 0 && col_ok && (rr.cnt > 0 || !rr.accumulate) ? C + (size_t)rr.row * n + col_off : nullptr;
#pragma unroll
            for (int x = 0; x < VEC; ++x) result[x] = rr.cnt > 0 ? acc[x] : A(0);
            buf ^= 1;
        }
        if (last) break;
        chunk = after;
        w0 = after_w0;
        wn = after_wn;
        rec ^= 1;
    }
    write_result();
}

template <typename T, int TILES>
__global__ void __launch_bounds__(kResThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
spmm_ring_kernel(int m2, int n, int slices, int owned_slots, bool all_windows, const int* __restrict__ plan, const int* __restrict__ col, const typename DenseVec<T>::Acc* __restrict__ val,
                 const T* __restrict__ B, typename DenseVec<T>::Acc* __restrict__ C, const PlannedChunk* __restrict__ rows)
{
    using A = typename DenseVec<T>::Acc;
    using R = Ring<TILES>;
    constexpr int VEC = DenseVec<T>::kElems, TW = kResLanes * VEC, QUADS = kBlockItems / 4;
    __shared__ uint4 ring[R::kBytes / 16];
    __shared__ uint4 records[3 * kRingRecordVecs];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int group = threadIdx.x / kResLanes, ls = threadIdx.x % kResLanes;
    __shared__ int walk_room[kResThreads / kWave + 2];
    const RingWalk walk(m2, slices, all_windows, plan, walk_room);
    int chunk = walk.from(rows, walk.at);
    if (chunk >= walk.end) return;
    const char* ring_bytes = reinterpret_cast<const char*>(ring);
    const unsigned ring_lds = lds_address(ring), rec_lds = lds_address(records), row_bytes = (unsigned)n * (unsigned)sizeof(T);
    const char* dense = reinterpret_cast<const char*>(B) + walk.slice * R::kRowBytes;
    const int col0 = walk.slice * TILES * TW + ls * VEC; // this lane's first column of B

    auto fetch_rows = [&](int from, int to) __attribute__((always_inline)) { R::fetch(ring_lds, dense, row_bytes, from, to, wave, lane); };
    auto fetch_record = [&](int rec, int c) __attribute__((always_inline)) { fetch_ring_record(rec_lds + rec * kRingRecordVecs * 16, rows + c, wave); };
    auto record = [&](int rec) __attribute__((always_inline)) -> const RingRecord& { return *reinterpret_cast<const RingRecord*>(records + rec * kRingRecordVecs); };
    // a row's values lie in the quads of its group: position 4 q + j in lane j
    const int lane_of_quad = ls % 4;
    auto own_values = [&](const RingRecord& rc, A (&v)[QUADS]) __attribute__((always_inline)) {
        const int4 meta = *reinterpret_cast<const int4*>(&rc.meta[group]);
#pragma unroll
        for (int q = 0; q < QUADS; ++q) {
            const int pos = 4 * q + lane_of_quad;
            v[q] = meta.x >= 0 && pos < (meta.z & 0xff) ? val[meta.y + ((rc.entry[group][pos] >> 9) & (kBlockItems - 1))] : A(0);
        }
    };

    int w0 = rows[chunk].w0, low = w0, high = w0 + rows[chunk].wn; // (the ring has rows [low, high))
    int after = walk.from(rows, chunk + 1), rec = 0;
    fetch_rows(low, high);
    fetch_record(0, chunk);
    if (after < walk.end) fetch_record(1, after);
    copies_done();
    __syncthreads();
    A v_next[QUADS];
    own_values(record(0), v_next);
    // a chunk's results, written during the next one: nobody waits for the stores then
    A result[TILES][VEC];
    A* result_at = nullptr;
    bool result_adds = false;
    auto write_result = [&]() __attribute__((always_inline)) {
        if (result_at == nullptr) return;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if (result_adds) {
#pragma unroll
                for (int x = 0; x < VEC; ++x) atomicAdd(result_at + t * TW + x, result[t][x]);
            } else {
                store_row<VEC>(result_at + t * TW, result[t]);
            }
        }
    };

    while (true) {
        copies_done();
        __syncthreads(); // the chunk's rows and the next one's record are in LDS, and every wave is done with the chunk before
        const RingRecord& mine = record(rec);
        const int4 meta = *reinterpret_cast<const int4*>(&mine.meta[group]);
        const bool listed = meta.x >= 0 && !(((meta.z >> 8) & 1) && ((meta.z >> 16) & 0xffff) <= owned_slots);
        const int cnt = listed ? meta.z & 0xff : 0;
        const unsigned missmask = listed ? (unsigned)meta.w : 0u;
        const bool accumulate = (meta.z >> 8) & 1;
        unsigned at[kBlockItems / 2];
#pragma unroll
        for (int i = 0; i < kBlockItems / 8; ++i) {
            const uint4 e = reinterpret_cast<const uint4*>(mine.entry[group])[i];
            at[4 * i] = R::units(e.x, w0, ls), at[4 * i + 1] = R::units(e.y, w0, ls), at[4 * i + 2] = R::units(e.z, w0, ls), at[4 * i + 3] = R::units(e.w, w0, ls);
        }
        const int wave_quads = wave_max_quads((cnt + 3) / 4);
        const bool wave_all_hit = __ballot(missmask != 0) == 0ull;
        A v[QUADS];
#pragma unroll
        for (int q = 0; q < QUADS; ++q) {
            v[q] = v_next[q];
            asm volatile("" : "+v"(v[q])); // waited for here, before the copies below
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
            own_values(record(rec1), v_next);
        }
        write_result();
        __builtin_amdgcn_sched_barrier(0); // the loads above are issued before the work below, not after it
        A acc[TILES][VEC];
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int x = 0; x < VEC; ++x) acc[t][x] = A(0);
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
                        if ((missmask >> (4 * q + j)) & 1u) { // outside the window: the row of B from memory
                            const int c = col[meta.y + ((mine.entry[group][4 * q + j] >> 9) & (kBlockItems - 1))];
#pragma unroll
                            for (int t = 0; t < TILES; ++t) raw[t][j] = *reinterpret_cast<const uint4*>(B + (size_t)c * n + col0 + t * TW);
                        }
                }
                const A v4[4] = {of_quad<0>(v[q]), of_quad<1>(v[q]), of_quad<2>(v[q]), of_quad<3>(v[q])};
#pragma unroll
                for (int t = 0; t < TILES; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        A b[VEC];
                        unpack_dense<T>(raw[t][j], b);
#pragma unroll
                        for (int x = 0; x < VEC; ++x) acc[t][x] = fma(v4[j], b[x], acc[t][x]);
                    }
            }
        }
        // a listed row without slots of its own (empty, unaligned start) is stored as zeros
        result_adds = accumulate;
        result_at = listed && (cnt > 0 || !accumulate) ? C + (size_t)meta.x * n + col0 : nullptr;
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int x = 0; x < VEC; ++x) result[t][x] = cnt > 0 ? acc[t][x] : A(0);
        if (last) break;
        if (!ahead) {
            __syncthreads(); // (the rows of a window that lies apart, in the place of this one's)
            fetch_rows(next_w0, next_end);
            low = next_w0, high = next_end;
        }
        w0 = next_w0, rec = rec1, after = after2;
    }
    write_result();
}

} // namespace

// The window kernel over the planned chunks of the residue list, for dense rows that window_takes.
template <typename T>
hipError_t spmm_window_launch(int m2, int n, int owned_slots, const int* col, const typename SpmmAcc<T>::type* val, const T* B,
                              typename SpmmAcc<T>::type* C, const PlanRef& plan, hipStream_t stream)
{
    if (m2 <= 0) return hipSuccess;
    const size_t row_bytes = (size_t)n * sizeof(T);
    const PlannedChunk* rows = static_cast<const PlannedChunk*>(plan.rows);
    if (plan.rings) {
        if (ring_slices(row_bytes) == 0) return hipErrorInvalidValue;
        const bool all = plan.host_counts != nullptr && plan.host_counts[1] == plan.host_counts[0];
        auto kernel = row_bytes == 128 ? spmm_ring_kernel<T, 1> : spmm_ring_kernel<T, 2>;
        kernel<<<kWindowWgs, kResThreads, 0, stream>>>(m2, n, ring_slices(row_bytes), owned_slots, all, plan.dev, col, val, B, C, rows);
        return hipGetLastError();
    }
    if (!window_takes(row_bytes)) return hipErrorInvalidValue;
    auto kernel = ((size_t)n * sizeof(T)) % (kResLanes * 16) != 0 ? spmm_residue_window_kernel<T, true> : spmm_residue_window_kernel<T, false>;
    kernel<<<window_grid(m2), kResThreads, 0, stream>>>(m2, n, owned_slots, col, val, B, C, rows);
    return hipGetLastError();
}

template hipError_t spmm_window_launch<float>(int, int, int, const int*, const float*, const float*, float*, const PlanRef&, hipStream_t);
template hipError_t spmm_window_launch<double>(int, int, int, const int*, const double*, const double*, double*, const PlanRef&, hipStream_t);
template hipError_t spmm_window_launch<__half>(int, int, int, const int*, const float*, const __half*, float*, const PlanRef&, hipStream_t);

} // namespace rode
