// Candidates of the kNN graph on the f16 matrix pipe (squared L2; the inner product and rows beyond 128 dimensions in whole
// chunks of 32).
//
// The graph is exact: what comes out of the matrix instructions are candidate lists, and knn_finish_kernel scores these in
// fp32 in the canonical order and proves, row by row, that no other column can belong into the row.  So the products may
// be rounded as long as the proof is told by how much.  Here a row is rounded to f16 once (eleven bits of what is left
// after centring), and the distance that the matrix instructions form is the distance between the ROUNDED rows, exact
// but for its fp32 sums: the products of two f16 values are exact in fp32.  How far a row moved when it was rounded is
// measured (eps, the norm of the remainder), and by the triangle inequality the distance of two rows is off by at most
// the sum of their two eps.  One instruction a product, where two bf16 halves a value take three and bound the error by
// the norms of the rows, not by their distance: at 1M x 128 the sweep went from 402 to 118 ms.  Rows of integers up to
// 2048 in magnitude do not move at all (the centre is rounded to a grid on which they stay integers): eps = 0.
//
// The inner product takes the same way without a centre: it is off by at most eps_i |c| + |q| eps_c.
//
//   1. centre and scale: a mean of spaced rows, a power of two that brings the longest row to [2^12, 2^13)
//   2. bounds: every row against an evenly spaced sample of the rows; a row's bound is about its distance to the rank-th
//      nearest sample row, so that a few hundred columns lie within it
//   3. rows in descending order of their bounds (half_order), packed once more in that order
//   4. sym_half_kernel, sym_half_long_kernel: each pair of rows once; a pair within a row's bound goes to that row's list
//   5. knn_finish_kernel: lists to neighbours, and the rows whose lists prove nothing
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "device_utils.hpp"
#include "half_rows.hpp"
#include "topk_gemm.hpp"
#include "topk_internal.hpp"

namespace grab {

using namespace dev;

namespace {

constexpr int kSampleClasses = 128;       // classes of sample columns (place mod 128) that keep a best value each
constexpr uint32_t kTileRows = 256;       // rows of a workgroup of sym_half_kernel
constexpr uint32_t kOrderBits = 14, kOrderBins = 1u << kOrderBits;


// the same for every place, where the sweep stages rows through LDS: 2 KB a block, the second KB zeros.  t: a threshold per
// place, or null
__global__ void __launch_bounds__(256) half_row_fragments_kernel(const float* __restrict__ hn, const float* __restrict__ t, float norm_factor,
                                                                 uint32_t places, uint4* __restrict__ out) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= places) return;
    uint4* o = out + (size_t)(p >> 5) * 128 + (p & 31);
    const float h = hn[p];
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    o[0] = row_norm_pieces(h >= 0.0f ? norm_factor * h - (t ? t[p] : 0.0f) : kNever * kNormUnit);
    o[32] = o[64] = o[96] = zero;
}

// Order of a block's instructions: column fragments are read from LDS two ahead of the matrix instructions that take them.
// (Left to itself the compiler keeps one in registers, and every pair of matrix instructions waits for a trip to LDS.)
template <int KS>
__device__ __forceinline__ void columns_ahead() {
    constexpr int AHEAD = 3;
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
    for (int ks = 0; ks <= KS; ++ks) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        if (ks + AHEAD <= KS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
}

// The same for a chunk of two fragments a block, 2 row and CB column blocks a wave: the second fragments are read while the
// first ones are multiplied.  100,003 x 768, inner product, the build: 23.77 -> 23.54 ms.
template <int CB>
__device__ __forceinline__ void chunk_ahead() {
    __builtin_amdgcn_sched_group_barrier(0x100, 2 + CB, 0);
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        if (2 * cb < 2 + CB) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 2 * CB, 0);
}

// Bounds.  A workgroup of four waves sets 128 rows against all sample columns, 64 a step; wave (wr, wc) owns 64 rows and 32
// columns of a step: a column's fragment, read from LDS, feeds two matrix instructions.  Every accumulator position keeps
// the largest value it sees, apart for even and odd steps: 128 classes of columns, 128 values a row, and the q-th largest
// of these stands in for the rank-th largest of all (half_bound_kernel).  Accumulator register v of lane (l32, half): row
// (v & 3) + 8 (v >> 2) + 4 half of the block, column l32.
template <int KS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) half_bound_sweep_kernel(const uint4* __restrict__ rows, const float* __restrict__ hn, float norm_factor, uint32_t n,
                                                                const uint4* __restrict__ sample, uint32_t steps, float* __restrict__ best) {
    constexpr uint32_t NP = 2 * (KS + 1), PF = (NP + 3) / 4;
    __shared__ v4u s_cols[2][NP * 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wr = wave >> 1, wc = wave & 1, half = lane >> 5, l32 = lane & 31;
    const uint32_t row0 = blockIdx.x * 128 + wr * 64;
    v8h a[2][KS + 1];
#pragma unroll
    for (uint32_t rb = 0; rb < 2; ++rb) {
        const uint4* src = rows + (size_t)(row0 / 32 + rb) * (KS + 1) * 64 + lane;
#pragma unroll
        for (uint32_t ks = 0; ks < KS; ++ks) a[rb][ks] = __builtin_bit_cast(v8h, src[ks * 64]);
        a[rb][KS] = row_norm_fragment(norm_factor * hn[row0 + rb * 32 + l32], half);
    }
    v16f most[2][2];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int v = 0; v < 16; ++v) most[q][rb][v] = -__builtin_inff();
    v4u st[PF];
    auto fetch = [&](uint32_t step) {
        const v4u* src = reinterpret_cast<const v4u*>(sample) + (size_t)min(step, steps - 1u) * NP * 64 + lane;
#pragma unroll
        for (uint32_t i = 0; i < PF; ++i) st[i] = src[min(wave + 4 * i, NP - 1) * 64];
    };
    auto park = [&](uint32_t buf) {
#pragma unroll
        for (uint32_t i = 0; i < PF; ++i) s_cols[buf][min(wave + 4 * i, NP - 1) * 64 + lane] = st[i];  // the same words where waves meet
    };
    fetch(0);
    park(0);
    fetch(1);
    __syncthreads();
    for (uint32_t step = 0; step < steps; step += 2) {  // steps is even
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q) {
            park(q ^ 1u);  // the buffer that everyone was through with before the barrier
            fetch(step + q + 2);
            const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            v16f acc0 = zero, acc1 = zero;
#pragma unroll
            for (uint32_t ks = 0; ks <= KS; ++ks) {
                const v8h b = __builtin_bit_cast(v8h, s_cols[q][(wc * (KS + 1) + ks) * 64 + lane]);
                acc0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][ks], b, acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][ks], b, acc1, 0, 0, 0);
            }
            columns_ahead<KS>();
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                most[q][0][v] = acc0[v] > most[q][0][v] ? acc0[v] : most[q][0][v];
                most[q][1][v] = acc1[v] > most[q][1][v] ? acc1[v] : most[q][1][v];
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q)
#pragma unroll
        for (uint32_t rb = 0; rb < 2; ++rb)
#pragma unroll
            for (uint32_t v = 0; v < 16; ++v) {
                const uint32_t row = row0 + rb * 32 + (v & 3) + 8 * (v >> 2) + 4 * half;
                if (row < n) best[(size_t)row * kSampleClasses + q * 64 + wc * 32 + l32] = most[q][rb][v];
            }
}

// bound[row]: the q-th largest of the row's 128 values, as a distance; a wave a row
__global__ void __launch_bounds__(256) half_bound_kernel(const float* __restrict__ best, const float* __restrict__ hn, const uint32_t* __restrict__ scal,
                                                         uint32_t n, uint32_t q, int ip, float* __restrict__ bound) {
    __shared__ __align__(16) float s_v[4][kSampleClasses];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t row = blockIdx.x * 4 + wave;
    if (row >= n) return;  // whole waves; no barrier below
    const float a = best[(size_t)row * kSampleClasses + lane], b = best[(size_t)row * kSampleClasses + 64 + lane];
    s_v[wave][lane] = a;
    s_v[wave][64 + lane] = b;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // place of a value = values that are larger, or equal at a lower index
    uint32_t ra = 0, rb = 0;
    const float4* v4 = reinterpret_cast<const float4*>(s_v[wave]);
#pragma unroll 4
    for (uint32_t c = 0; c < kSampleClasses / 4; ++c) {
        const float4 v = v4[c];
        const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t at = 4 * c + u;
            ra += (e[u] > a || (e[u] == a && at < lane)) ? 1u : 0u;
            rb += (e[u] > b || (e[u] == b && at < 64 + lane)) ? 1u : 0u;
        }
    }
    const float s = scale_of(__uint_as_float(scal[0])), unit = (ip ? -1.0f : -2.0f) / (s * s), least = ip ? -__builtin_inff() : 0.0f;
    const bool good = hn[row] >= 0.0f;  // a row that is not finite gets no list
    if (ra == q - 1) bound[row] = good ? fmaxf(a * unit, least) : 0.0f;
    if (rb == q - 1) bound[row] = good ? fmaxf(b * unit, least) : 0.0f;
}

// ---- rows in descending order of their bounds ------------------------------------------------------------------
// The sweep asks of a pair (i, j) whether it lies within either row's bound.  With the rows in descending order of their
// bounds and j behind i, the larger one is i's, always: one threshold, known before the sweep, which goes into the row's norm
// fragment, and the test of a pair is the sign of its accumulator.  The order is by the upper 14 bits of the bound (steps of
// 3 %); within a step the rows share its upper edge as their threshold, and their own bounds are looked at where a pair
// passed.
__device__ __forceinline__ uint32_t order_bin(float bound) { return kOrderBins - 1u - (ord_bits(bound) >> (32 - kOrderBits)); }
__device__ __forceinline__ float bin_edge(float bound) { return ord_float(ord_bits(bound) | ((1u << (32 - kOrderBits)) - 1u)); }

constexpr uint32_t kOrderRows = 8192;  // rows of a workgroup
__global__ void __launch_bounds__(1024) order_count_kernel(const float* __restrict__ bound, uint32_t n, uint32_t* __restrict__ bins) {
    extern __shared__ uint32_t s_bins[];
    for (uint32_t b = threadIdx.x; b < kOrderBins; b += 1024) s_bins[b] = 0;
    __syncthreads();
    const uint32_t end = min(n, (blockIdx.x + 1) * kOrderRows);
    for (uint32_t i = blockIdx.x * kOrderRows + threadIdx.x; i < end; i += 1024) atomicAdd(&s_bins[order_bin(bound[i])], 1u);
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < kOrderBins; b += 1024)
        if (s_bins[b] != 0) atomicAdd(&bins[b], s_bins[b]);
}
__global__ void __launch_bounds__(1024) order_scan_kernel(uint32_t* __restrict__ bins) {  // counts become first places
    __shared__ uint32_t s_sum[1024];
    constexpr uint32_t PER = kOrderBins / 1024;
    uint32_t v[PER], sum = 0;
#pragma unroll
    for (uint32_t u = 0; u < PER; ++u) {
        v[u] = bins[threadIdx.x * PER + u];
        sum += v[u];
    }
    s_sum[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t w = 1; w < 1024; w <<= 1) {
        const uint32_t before = threadIdx.x >= w ? s_sum[threadIdx.x - w] : 0u;
        __syncthreads();
        s_sum[threadIdx.x] += before;
        __syncthreads();
    }
    uint32_t at = s_sum[threadIdx.x] - sum;
#pragma unroll
    for (uint32_t u = 0; u < PER; ++u) {
        bins[threadIdx.x * PER + u] = at;
        at += v[u];
    }
}
__global__ void __launch_bounds__(1024) order_place_kernel(const float* __restrict__ bound, uint32_t n, uint32_t* __restrict__ bins,
                                                         uint32_t* __restrict__ perm) {
    extern __shared__ uint32_t s_bins[];
    for (uint32_t b = threadIdx.x; b < kOrderBins; b += 1024) s_bins[b] = 0;
    __syncthreads();
    const uint32_t begin = blockIdx.x * kOrderRows, end = min(n, begin + kOrderRows);
    uint32_t bin[kOrderRows / 1024], at[kOrderRows / 1024];
#pragma unroll
    for (uint32_t u = 0; u < kOrderRows / 1024; ++u) {
        const uint32_t i = begin + u * 1024 + threadIdx.x;
        if (i < end) {
            bin[u] = order_bin(bound[i]);
            at[u] = atomicAdd(&s_bins[bin[u]], 1u);
        }
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < kOrderBins; b += 1024)
        if (s_bins[b] != 0) s_bins[b] = atomicAdd(&bins[b], s_bins[b]);
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < kOrderRows / 1024; ++u) {
        const uint32_t i = begin + u * 1024 + threadIdx.x;
        if (i < end) perm[s_bins[bin[u]] + at[u]] = i;
    }
}
// per place: the row's threshold and its step's, on the accumulators' scale (minus half a squared distance, or the inner
// product), and the largest value there can be
__global__ void __launch_bounds__(256) order_thresholds_kernel(const float* __restrict__ bound, const uint32_t* __restrict__ perm, const uint32_t* __restrict__ scal,
                                                               const float* __restrict__ hn, uint32_t n, uint32_t places, int ip, float* __restrict__ t_own,
                                                               float* __restrict__ t_step, float* __restrict__ top) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= places) return;
    const float s = scale_of(__uint_as_float(scal[0])), unit = (ip ? -1.0f : -0.5f) * (s * s), b = p < n ? bound[perm[p]] : 0.0f;
    t_own[p] = p < n ? b * unit : __builtin_inff();
    t_step[p] = p < n ? bin_edge(b) * unit : 0.0f;
    top[p] = ip ? sqrtf(fmaxf(hn[p], 0.0f)) * 8192.0f : 0.0f;
}

// ---- the sweep ---------------------------------------------------------------------------------------------------
// Workgroup = 4 waves, three workgroups a CU (four up to 64 dimensions: half_groups); a workgroup owns 256 rows and sweeps the columns from the last one back to
// its own rows, 32 a step.  Wave w owns rows 64 w .. + 63: their fragments stay in registers for the whole sweep (72 for
// 128 dimensions), and a column's fragment, read from LDS, feeds two matrix instructions - 64 bytes a cycle for the CU's
// four matrix pipes at full rate, half of what LDS delivers.  (32 rows a wave would need all of it.)  The columns of the
// next step but one travel in registers (5 x 16 bytes a lane) while a step runs; one barrier a step.
//
// The epilogue is made for pairs that do not matter, all but about one in a thousand: an accumulator holds -d/2 less the
// row's threshold, so the 16 values of a lane are of no use when all of them are negative - eight three-way integer maxima
// and a compare for a block of 32 x 32.  A lane that has a value above zero copies all 16 into a queue in LDS (four
// 16-byte writes, whichever lanes it is) and the sweep goes on.  When 16 such entries have gathered the wave goes over
// them, 64 values at a time, packs the pairs that passed and appends them, 64 at a time, to the rows' lists in device
// memory: the trips to memory (a place in the list of each row, then the key) are paid once for 64 pairs.
//
// What bounds it: the matrix pipes, busy 60 % of the launch's cycles at 1.9 GHz.  1M x 128: 1.44e14 operations in 118 ms, 1.2
// PFLOP/s, against 402 ms on two bf16 halves a value; without the queue (a variant that appends nothing) 94 ms, 1.5 PFLOP/s,
// where a large library product reaches 1.28 on the same card.  The columns come from L2: 0.15 TB fetched of 0.6 TB loaded.
// Two workgroups a CU with steps of 64 columns: 123 ms.
struct SymHalfArgs {
    const uint4* blocks;
    const uint4* row_frags;  // sym_half_long_kernel: the rows' norm fragments
    const float* hn;         // per place
    const float* t_own;
    const float* t_step;
    const float* top;
    const uint32_t* perm;  // place -> row
    uint32_t* list;        // [n][cap] entries per place (share_of)
    uint32_t id_bits;
    uint32_t* count;       // entries offered to a place (may exceed cap: its row is then redone the plain way)
    uint32_t cap, n;
    float norm_factor;
    uint32_t frags;        // of a block
    uint32_t row_tiles, steps, steps_per_slice, slices;  // steps: of 32 columns (long rows: of a tile's), of the whole row set
    uint32_t* work_counter;
};
struct RowTables {  // of a workgroup's 256 rows
    float t_own[kTileRows], t_step[kTileRows], top[kTileRows];
    uint32_t id[kTileRows];
};
struct SymSink {
    const SymHalfArgs& a;
    const RowTables& rows;
    uint32_t row0 = 0, rt = 0;  // first row of the workgroup, its tile
    __device__ __forceinline__ void put(float value, uint32_t il, uint32_t j) const {
        const uint32_t i = row0 + il;
        const float g = value + rows.t_step[il];
        uint32_t at_i = 0xFFFFFFFFu, at_j = 0xFFFFFFFFu;
        const float ti = rows.t_own[il];
        if (g >= ti && j < a.n) at_i = atomicAdd(&a.count[i], 1u);
        const float tj = a.t_own[j], top_j = a.top[j];
        const uint32_t id_j = a.perm[min(j, a.n - 1u)];
        // the diagonal tile holds both orders of its pairs itself
        if ((j / kTileRows) != rt && g >= tj) at_j = atomicAdd(&a.count[j], 1u);
        if (at_i < a.cap) a.list[(size_t)i * a.cap + at_i] = id_j | share_of(g, ti, rows.top[il], a.id_bits);
        if (at_j < a.cap) a.list[(size_t)j * a.cap + at_j] = rows.id[il] | share_of(g, tj, top_j, a.id_bits);
    }
};
template <int KS>
struct SymHalfLds {
    v4u cols[2][(KS + 1) * 64];
    QueueLds queue[4];
    RowTables rows;
    uint32_t next_item;
};

__device__ __forceinline__ void load_row_tables(const SymHalfArgs& a, RowTables& rows, uint32_t row0, uint32_t tid) {
    if (tid < kTileRows) {  // places are padded to whole tiles
        rows.t_own[tid] = a.t_own[row0 + tid];
        rows.t_step[tid] = a.t_step[row0 + tid];
        rows.top[tid] = a.top[row0 + tid];
        rows.id[tid] = row0 + tid < a.n ? a.perm[row0 + tid] : 0u;
    }
}

constexpr uint32_t half_groups(int ks) { return ks >= 6 ? 3u : 4u; }  // workgroups a CU: what registers and LDS allow
template <int KS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(half_groups(KS), half_groups(KS)))) sym_half_kernel(const SymHalfArgs a) {
    extern __shared__ __align__(16) uint8_t half_smem[];
    SymHalfLds<KS>& s = *reinterpret_cast<SymHalfLds<KS>*>(half_smem);
    constexpr uint32_t NP = KS + 1, PF = (NP + 3) / 4;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), half = lane >> 5, l32 = lane & 31;
    const uint32_t nwork = a.row_tiles * a.slices;
    PairQueue<SymSink> queue(SymSink{a, s.rows}, s.queue[wave], lane, wave * 64);

    for (;;) {
        __syncthreads();  // the item before is fully drained
        if (tid == 0) s.next_item = atomicAdd(a.work_counter, 1u);
        __syncthreads();
        const uint32_t work = (uint32_t)__builtin_amdgcn_readfirstlane((int)s.next_item);
        if (work >= nwork) break;  // workgroup-uniform
        const uint32_t slice = work / a.row_tiles, rt = work - slice * a.row_tiles, row0 = rt * kTileRows;
        // this item: the steps [begin, end) of 32 columns, from the last one down
        const uint32_t before = slice * a.steps_per_slice;
        if (before >= a.steps || a.steps - before <= rt * (kTileRows / 32)) continue;  // workgroup-uniform: below the diagonal
        const uint32_t end = a.steps - before, begin = max(rt * (kTileRows / 32), end > a.steps_per_slice ? end - a.steps_per_slice : 0u);
        load_row_tables(a, s.rows, row0, tid);
        queue.sink.row0 = row0;
        queue.sink.rt = rt;
        v8h af[2][KS + 1];
#pragma unroll
        for (uint32_t rb = 0; rb < 2; ++rb) {
            const uint32_t r = row0 + wave * 64 + rb * 32;
            const uint4* src = a.blocks + (size_t)(r / 32) * (KS + 1) * 64 + lane;
#pragma unroll
            for (uint32_t ks = 0; ks < KS; ++ks) af[rb][ks] = __builtin_bit_cast(v8h, src[ks * 64]);
            const float hn = a.hn[r + l32];
            af[rb][KS] = row_norm_fragment(hn >= 0.0f ? a.norm_factor * hn - a.t_step[r + l32] : kNever * kNormUnit, half);
        }

        v4u st[PF];
        auto fetch = [&](uint32_t step) {
            const v4u* src = reinterpret_cast<const v4u*>(a.blocks) + (size_t)step * NP * 64 + lane;
#pragma unroll
            for (uint32_t i = 0; i < PF; ++i) st[i] = src[min(wave + 4 * i, NP - 1) * 64];
        };
        auto park = [&](uint32_t buf) {
#pragma unroll
            for (uint32_t i = 0; i < PF; ++i) s.cols[buf][min(wave + 4 * i, NP - 1) * 64 + lane] = st[i];  // the same words where waves meet
        };
        // (past the end of the sweep the first step is fetched once more, into the buffer nobody reads)
        fetch(end - 1);
        park(0);
        fetch(end - 1 > begin ? end - 2 : begin);
        __syncthreads();  // first columns and row tables visible
        uint32_t buf = 0;
        for (uint32_t step = end; step-- > begin; buf ^= 1u) {
            park(buf ^ 1u);
            fetch(step >= begin + 2 ? step - 2 : begin);
            const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            v16f acc[2] = {zero, zero};
            const v4u* col = &s.cols[buf][lane];
#pragma unroll
            for (uint32_t ks = 0; ks <= KS; ++ks) {  // the norms last: they are added to the finished sum of products
                const v8h b = __builtin_bit_cast(v8h, col[ks * 64]);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[0][ks], b, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[1][ks], b, acc[1], 0, 0, 0);
            }
            columns_ahead<KS>();
            queue.offer(acc[0], step * 32 + l32, 0);
            queue.offer(acc[1], step * 32 + l32, 1);
            __syncthreads();  // everyone is through with these columns
        }
        queue.finish();
    }
}

// ---- the same sweep for longer rows ------------------------------------------------------------------------------
// Rows do not fit a wave's registers: rows and columns go through LDS, 32 dimensions (two fragments a block) at a time.  One
// workgroup of eight waves a CU, a tile of 256 rows x 64 CB columns; wave (wr, wc) owns 64 rows and 32 CB columns of it.  CB = 4,
// the sweep: six fragments from LDS feed eight matrix instructions, 96 bytes a cycle at full rate of the 128 there are.  CB =
// 2, BOUND: the bounds against the sample (half_bound_sweep_kernel), with the best values in the other half of the registers.
// The next chunk goes from memory straight into the other LDS buffer while one is multiplied; one barrier a chunk.  Items
// (row tile, slice of column tiles) are dealt out by XCD (next_long_item), so that the 32 workgroups that share an L2 read
// eight row tiles and four slices between them.
// What bounds it: LDS.  100,003 x 768, inner product: 7.7e12 operations in 10.5 ms, 0.74 PFLOP/s (26.3 ms on two bf16 halves a
// value, three instructions a product), matrix pipes busy 37 % of the cycles; a variant that loads nothing more takes 4.7 ms,
// near the pipes' own time: 96 KB read and 32 KB written a chunk are 1000 cycles of LDS beside 1024 of matrix instructions, and
// the two do not overlap to the end.  Through registers on the way to LDS 11.0 ms; two chunks under way instead of one the
// same; two workgroups of four waves on 256 x 128 each 11.4 ms.
constexpr uint32_t kLongXcds = 8, kLongGroup = 8;
template <int CB, bool BOUND>
struct SymLongLds {
    QueueLds queue[BOUND ? 1 : 8];
    RowTables rows;
    uint32_t next_item;
};
// the next (row tile, slice): row tile * slices + slice, all-ones when none is left.  A queue per XCD, in which the slices of
// eight row tiles follow each other; an empty queue's workgroups go on with the next XCD's.
__device__ __forceinline__ uint32_t next_long_item(const SymHalfArgs& a) {
    const uint32_t groups = (a.row_tiles + kLongGroup - 1) / kLongGroup, per_group = kLongGroup * a.slices;
    for (uint32_t t = 0; t < kLongXcds; ++t) {
        const uint32_t x = (blockIdx.x + t) % kLongXcds, items = groups > x ? (groups - x + kLongXcds - 1) / kLongXcds * per_group : 0u;
        for (;;) {
            const uint32_t i = atomicAdd(a.work_counter + x, 1u);
            if (i >= items) break;
            const uint32_t k = i / per_group, sl = (i - k * per_group) / kLongGroup, rt = (x + k * kLongXcds) * kLongGroup + i % kLongGroup;
            if (rt < a.row_tiles && rt + sl * a.steps_per_slice < a.steps) return rt * a.slices + sl;
        }
    }
    return 0xFFFFFFFFu;
}

template <int CB, bool BOUND>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
sym_half_long_kernel(const SymHalfArgs a, const uint4* __restrict__ columns, float* __restrict__ best) {
    extern __shared__ __align__(16) uint8_t half_smem[];
    SymLongLds<CB, BOUND>& s = *reinterpret_cast<SymLongLds<CB, BOUND>*>(half_smem);
    constexpr uint32_t kLongRows = kTileRows / 32 * 128, kChunk = kLongRows + CB * 2 * 128;
    // two variables, not two halves of one: the compiler must see that the reads of one do not wait for the loads into the other
    __shared__ v4u s_chunk0[kChunk], s_chunk1[kChunk];
    constexpr uint32_t kThreads = 512, kCols = 64 * CB, AF = kTileRows / 32 * 128 / kThreads, BF = CB * 2 * 128 / kThreads;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), half = lane >> 5, l32 = lane & 31;
    const uint32_t wr = wave >> 1, wc = wave & 1, chunks = a.frags / 2;
    PairQueue<SymSink> queue(SymSink{a, s.rows}, s.queue[BOUND ? 0 : wave], lane, wr * 64);
    for (;;) {
        loads_landed();   // the one too many that the item before has under way, also before the workgroup ends
        __syncthreads();  // the item before is fully drained
        if (tid == 0) s.next_item = BOUND ? atomicAdd(a.work_counter, 1u) : next_long_item(a);
        __syncthreads();
        const uint32_t work = (uint32_t)__builtin_amdgcn_readfirstlane((int)s.next_item);
        if (work >= a.row_tiles * a.slices) break;  // workgroup-uniform
        const uint32_t rt = work / a.slices, slice = work - rt * a.slices, row0 = rt * kTileRows;
        // column tiles [begin, end), from the last one down; the sweep's not below the diagonal
        const uint32_t end = a.steps - slice * a.steps_per_slice;
        const uint32_t begin = max(BOUND ? 0u : rt, end > a.steps_per_slice ? end - a.steps_per_slice : 0u);
        if (!BOUND) load_row_tables(a, s.rows, row0, tid);
        queue.sink.row0 = row0;
        queue.sink.rt = rt;

        // chunk c of the rows and of column tile ct, straight into LDS: two fragments of every block, 2 KB in a row, 1 KB a wave
        // and instruction
        auto load = [&](v4u* to, uint32_t ct, uint32_t c) {
            const bool norms = c + 1 >= chunks;  // workgroup-uniform
            c = min(c, chunks - 1u);
            const v4u* ra = reinterpret_cast<const v4u*>(norms ? a.row_frags : a.blocks);
            const uint32_t pitch = norms ? 128u : a.frags * 64, from = norms ? 0u : c * 128;
#pragma unroll
            for (uint32_t i = 0; i < AF; ++i) {
                const uint32_t at = tid + kThreads * i;
                load_to_lds(ra + (size_t)(row0 / 32 + (at >> 7)) * pitch + from + (at & 127u), to + wave * 64 + kThreads * i);
            }
            const v4u* rb = reinterpret_cast<const v4u*>(columns) + (size_t)ct * (kCols / 32) * a.frags * 64 + c * 128;
#pragma unroll
            for (uint32_t i = 0; i < BF; ++i) {
                const uint32_t at = tid + kThreads * i;
                load_to_lds(rb + (size_t)(at >> 7) * a.frags * 64 + (at & 127u), to + kLongRows + wave * 64 + kThreads * i);
            }
        };
        const uint32_t padded = (chunks + 1u) & ~1u;  // chunks go in pairs; nothing is multiplied in one too many
        uint32_t ct = end - 1, c = 0, ct_next = ct, c_next = 0;  // what is multiplied, and what was asked for last
        auto advance = [&]() {  // (past the end of the item the last chunk is fetched once more, into the buffer nobody reads)
            if (++c_next == padded) {
                if (ct_next > begin) {
                    --ct_next;
                    c_next = 0;
                } else {
                    c_next = padded - 1;
                }
            }
        };
        v16f most[BOUND ? 2 : 1][BOUND ? CB : 1];
        if (BOUND) {
#pragma unroll
            for (uint32_t rb = 0; rb < (BOUND ? 2 : 1); ++rb)
#pragma unroll
                for (uint32_t cb = 0; cb < (BOUND ? CB : 1); ++cb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) most[rb][cb][v] = -__builtin_inff();
        }
        v16f acc[2][CB];
        auto multiply = [&](const v4u* from, auto first_chunk) {
            constexpr bool FIRST = decltype(first_chunk)::value;
            const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t ks = 0; ks < 2; ++ks) {
                v8h x[2], y[CB];
#pragma unroll
                for (uint32_t rb = 0; rb < 2; ++rb) x[rb] = __builtin_bit_cast(v8h, from[(wr * 2 + rb) * 128 + ks * 64 + lane]);
#pragma unroll
                for (uint32_t cb = 0; cb < CB; ++cb) y[cb] = __builtin_bit_cast(v8h, from[kLongRows + (wc * CB + cb) * 128 + ks * 64 + lane]);
#pragma unroll
                for (uint32_t cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (uint32_t rb = 0; rb < 2; ++rb)
                        acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[rb], y[cb], FIRST && ks == 0 ? zero : acc[rb][cb], 0, 0, 0);
            }
            chunk_ahead<CB>();
        };
        load(s_chunk0, ct_next, c_next);
        loads_landed();
        __syncthreads();  // first chunk and row tables visible
        for (;;) {
            advance();
            load(s_chunk1, ct_next, c_next);
            if (c == 0) multiply(s_chunk0, std::true_type{});
            else multiply(s_chunk0, std::false_type{});
            loads_landed();
            __syncthreads();  // everyone is through with this chunk, the next one is there
            advance();
            load(s_chunk0, ct_next, c_next);
            if (c + 1 < chunks) multiply(s_chunk1, std::false_type{});
            c += 2;
            if (c == padded) {
                const uint32_t col = ct * kCols + wc * (32 * CB) + l32;
#pragma unroll
                for (uint32_t cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (uint32_t rb = 0; rb < 2; ++rb) {
                        if (BOUND) {
                            v16f& m = most[BOUND ? rb : 0][BOUND ? cb : 0];
#pragma unroll
                            for (int v = 0; v < 16; ++v) m[v] = acc[rb][cb][v] > m[v] ? acc[rb][cb][v] : m[v];
                        } else {
                            queue.offer(acc[rb][cb], col + cb * 32, rb);
                        }
                    }
                if (ct == begin) break;  // workgroup-uniform
                --ct;
                c = 0;
            }
            loads_landed();
            __syncthreads();
        }
        if (BOUND) {
#pragma unroll
            for (uint32_t rb = 0; rb < (BOUND ? 2 : 1); ++rb)
#pragma unroll
                for (uint32_t cb = 0; cb < (BOUND ? CB : 1); ++cb)
#pragma unroll
                    for (uint32_t v = 0; v < 16; ++v) {
                        const uint32_t row = row0 + wr * 64 + rb * 32 + (v & 3) + 8 * (v >> 2) + 4 * half;
                        if (row < a.n) best[(size_t)row * kSampleClasses + wc * 64 + cb * 32 + l32] = most[rb][cb][v];
                    }
        } else {
            queue.finish();
        }
    }
}

// ---- lists to neighbours -------------------------------------------------------------------------------------------
// One wave per place.  Of the row's list - every column whose distance between the rounded rows is within the bound - those
// that can be among the k nearest (k + 1 with the row itself) are scored in the canonical order, sorted by (distance, id)
// and written; a row whose list does not prove the result is listed for another pass.
//   How far a distance can be off, squared L2: with D the distance (not squared) between two rounded rows, the true one lies
// within D +- (eps_i + eps_max); the squared value that the matrix instructions left is off the squared D by at most
// `form` = the fp32 sums' rounding - dim products, the norms' pieces and the threshold, twice should the pipe chop - relative
// to the norms.  Inner product: within eps_i |c| + (|q| + eps_i) eps_max + form of the product of the rows.  The fp32 GEMM
// form over the rows as they are, which a redone row may go through, has its own; the larger one is taken for both, so that
// a row is proven here or there alike.
struct FinishArgs {
    const float* data;
    const uint32_t* list;
    const uint32_t* count;
    const uint32_t* perm;
    const float* bound;   // per row
    const float* t_own;   // per place: the bound and the largest value, on the accumulators' scale
    const float* top;
    const float* norm;    // squared norms of the rows, and the largest
    const float* max_norm;
    const float* cnorm;   // ... of the centred rows; the largest is scal[0]
    const float* eps;     // the largest is scal[1]
    const uint32_t* scal;
    uint32_t* out;        // [n][k]
    uint32_t* redo_count;  // rows whose list is too short or too long, or the bound too near
    uint32_t* redo;
    uint32_t* doubt;      // [0] how many, then the rows: distances below what the forms resolve
    uint32_t n, dim, k, cap, min_list, id_bits;
    uint32_t redo_keep;   // candidates that the plain pass keeps for a row
};
constexpr uint32_t kFinishCap = 1024;
template <int METRIC>
__global__ void __launch_bounds__(256) knn_finish_kernel(const FinishArgs a) {
    __shared__ uint64_t keys_all[4][kFinishCap];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t p = blockIdx.x * 4 + wave;
    if (p >= a.n) return;  // wave-uniform; no barrier below
    uint64_t* keys = keys_all[wave];
    const uint32_t row = a.perm[p], have = a.count[p], need = a.k;  // the k-th of the keys from 0 on: k and the row itself
    if (have > a.cap || have < a.min_list) {
        if (lane == 0) a.redo[atomicAdd(a.redo_count, 1u)] = row;
        return;
    }
    uint32_t ent[16];
    const uint32_t* mine = a.list + (size_t)p * a.cap;
#pragma unroll
    for (int i = 0; i < 16; ++i) ent[i] = (uint32_t)(i * 64 + lane) < have ? mine[i * 64 + lane] : kInvalidId;
    auto within = [&](uint32_t part) {  // entries in the bound's parts up to `part`
        uint32_t c = 0;
        const uint32_t last = (part << a.id_bits) | ((1u << a.id_bits) - 1u);
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if ((uint32_t)(i * 64) < have) c += (uint32_t)__popcll(__ballot((uint32_t)(i * 64 + lane) < have && ent[i] <= last));
        return c;
    };
    // a part that need + 1 entries lie in or below, and few more
    const uint32_t parts = 1u << (32u - a.id_bits);
    uint32_t low = 0, high = parts - 1u, n_high = have;  // have > need
    while (low < high && n_high > need + 4) {
        const uint32_t mid = (low + high) >> 1, c = within(mid);
        if (c > need) {
            high = mid;
            n_high = c;
        } else {
            low = mid + 1;
        }
    }
    const double u = 5.9604644775390625e-08, dim = a.dim, rescore = (a.dim / 8 + 8) * u;
    const double eps = a.eps[row], eps_max = __uint_as_float(a.scal[1]), cn = a.cnorm[row], cn_max = __uint_as_float(a.scal[0]);
    const double bound = (double)a.bound[row];
    const double scale = scale_of(__uint_as_float(a.scal[0])), unit = (METRIC == kMetricL2 ? -2.0 : -1.0) / (scale * scale);
    // l2: what a distance can be off besides form; ip: what a product can be off in all
    double form, e_far;
    if (METRIC == kMetricL2) {
        form = fmax((3.25 * dim + 96.0) * u * (cn + cn_max), (1.25 * dim + 16.0) * u * ((double)a.norm[row] + (double)*a.max_norm));
        e_far = eps + eps_max;
    } else {
        form = fmax((2.0 * dim + 96.0) * u * sqrt(cn * cn_max), 2.0 * (1.25 * dim + 16.0) * u * sqrt((double)a.norm[row] * (double)*a.max_norm));
        e_far = eps * sqrt(cn_max) + (sqrt(cn) + eps) * eps_max + form;
    }
    if (a.scal[kScalLong] != 0) form = __builtin_inf();  // a row that is in no list, and may be near this one: nothing is proven
    // need + 1 columns' values lie in the parts up to `high`: their true distances lie within what the parts' lower edge, farthest
    // off, allows; a column whose value is beyond what follows from that is farther than all of them, also in the re-scored
    // order.  (A part's number was rounded: two parts more at either end.)
    const double top = a.top[p], way = top - (double)a.t_own[p], edge = (top - way * (high + 2.0) / parts) * unit;
    double cutoff;
    if (METRIC == kMetricL2) {
        const double reach = sqrt(edge + form) * (1.0 + 2.0 * rescore) + 2.0 * e_far;
        cutoff = reach * reach + form;
    } else {
        cutoff = edge + 2.0 * e_far + 2.0 * form;  // (the re-scoring's own error: `form` is no less)
    }
    const double far_part = (top - cutoff / unit) / way * parts + 1.0;
    const uint32_t last_part = far_part < (double)(parts - 1u) ? (uint32_t)fmax(far_part, 0.0) : parts - 1u;  // (all of them where it is not a number)
    uint32_t n_score = 0;
    {
        const uint32_t id_mask = (1u << a.id_bits) - 1u, last = (last_part << a.id_bits) | id_mask;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if ((uint32_t)(i * 64) < have) {
                const bool in = (uint32_t)(i * 64 + lane) < have && ent[i] <= last;
                const uint64_t b = __ballot(in);
                if (in) keys[n_score + (uint32_t)__popcll(b & ((1ull << lane) - 1ull))] = ent[i] & id_mask;
                n_score += (uint32_t)__popcll(b);
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // Bound by the latency of its gathers: two rows per group of 8 lanes at a time, eight 16-byte loads a lane in flight
    const float* q = a.data + (size_t)row * a.dim;
    const float4* q4 = reinterpret_cast<const float4*>(q);
    const int grp = lane >> 3, j = lane & 7;
    for (uint32_t c0 = 0; c0 < n_score; c0 += 16) {
        const uint32_t ca = c0 + grp, cb = ca + 8;
        if (ca >= n_score) continue;
        const uint32_t ia = (uint32_t)keys[ca], ib = cb < n_score ? (uint32_t)keys[cb] : ia;
        float da = 0.0f, db = 0.0f;
        fold_rows_any<METRIC, true>(reinterpret_cast<const float4*>(a.data + (size_t)ia * a.dim), reinterpret_cast<const float4*>(a.data + (size_t)ib * a.dim),
                                       q4, j, a.dim >> 2, da, db);
        da = group8_sum(da);
        db = group8_sum(db);
        if (j == 0) keys[ca] = make_sel_key(METRIC == kMetricIP ? -da : da, ia);
        if (j == 0 && cb < n_score) keys[cb] = make_sel_key(METRIC == kMetricIP ? -db : db, ib);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (n_score <= 256) {
        uint64_t k4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) k4[i] = (uint32_t)(lane * 4 + i) < n_score ? keys[lane * 4 + i] : kInvalidKey;
        wave_bitonic_sort<4>(k4);
#pragma unroll
        for (int i = 0; i < 4; ++i) keys[lane * 4 + i] = k4[i];
    } else {
        uint64_t k16[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) k16[i] = (uint32_t)(lane * 16 + i) < n_score ? keys[lane * 16 + i] : kInvalidKey;
        wave_bitonic_sort<16>(k16);
#pragma unroll
        for (int i = 0; i < 16; ++i) keys[lane * 16 + i] = k16[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    {   // every column that is not in the list lies at or beyond the bound
        const double last = (double)ord_float((uint32_t)(keys[need] >> 32));
        bool proven;
        if (METRIC == kMetricL2) {
            const double near_b = sqrt(fmax(bound - form, 0.0)) - e_far, out = near_b > 0.0 ? near_b * near_b : 0.0;
            proven = last < out - rescore * out;
        } else {
            proven = last < bound - e_far - form;
        }
        if (!proven) {  // (also where something is not a number)
            if (lane == 0) {
                // the plain pass has a form of its own, as far off: a longer list would hardly help
                bool hopeless = form > 0.005 * fabs(bound);
                if (METRIC == kMetricIP) {
                    // on bf16 halves it is off by half_err; how far its last candidate lies behind the k-th is reckoned from this list.  (Unit rows
                    // in tight clusters, 20,000 x 128: none of 20,000 was proven there, 29.3 ms a call with that pass, 22.4 before f16 rows)
                    const double half_err = 2.0 * (7.25 * dim + 816.0) * u * sqrt((double)a.norm[row] * (double)*a.max_norm);
                    const double more = have < a.redo_keep ? (double)(a.redo_keep - have) / (double)(have - need) : 0.0;
                    hopeless = hopeless || (bound - last) * (1.0 + more) < 0.5 * half_err;
                }
                if (hopeless) a.doubt[1 + atomicAdd(a.doubt, 1u)] = row;
                else a.redo[atomicAdd(a.redo_count, 1u)] = row;
            }
            return;
        }
    }
    // cagra.cu:181-196: skip the row's own id, keep k, pad with 0xFFFFFFFF
    uint32_t self_pos = 0xFFFFFFFFu;
    for (uint32_t base = 0; base <= need; base += 64) {
        const uint32_t g = base + lane;
        const bool is_self = g <= need && (uint32_t)keys[g] == row;
        const uint64_t b = __ballot(is_self);
        if (b != 0 && self_pos == 0xFFFFFFFFu) self_pos = base + (uint32_t)__builtin_ctzll(b);
    }
    for (uint32_t o = lane; o < a.k; o += 64) a.out[(size_t)row * a.k + o] = (uint32_t)keys[o + (o >= self_pos ? 1u : 0u)];
}

uint32_t ks_of(uint32_t dim) { return dim <= 32 ? 2 : dim <= 64 ? 4 : dim <= 96 ? 6 : dim <= 128 ? 8 : dim / 16; }
float norm_factor(const HalfKnn& h) { return h.ip ? 0.0f : -0.5f; }

SymHalfArgs sweep_args(const HalfKnn& h) {
    SymHalfArgs s{};
    s.blocks = h.blocks;
    s.row_frags = h.row_frags;
    s.hn = h.hn;
    s.t_own = h.t_own;
    s.t_step = h.t_step;
    s.top = h.top;
    s.perm = h.perm;
    s.list = h.list;
    s.id_bits = h.id_bits;
    s.count = h.count;
    s.cap = kHalfListCap;
    s.n = h.n;
    s.norm_factor = norm_factor(h);
    s.frags = h.frags;
    s.row_tiles = h.places / kTileRows;
    return s;
}

template <int KS>
int launch_bounds_short(const HalfKnn& h, hipStream_t st) {
    hipLaunchKernelGGL(half_bound_sweep_kernel<KS>, dim3(h.places / 128), dim3(256), 0, st, h.blocks, h.hn, norm_factor(h), h.n, h.sample_blocks,
                       h.sample_places / 64, h.best);
    return GRAB_OK;
}

template <int KS>
int launch_sweep_short(const HalfKnn& h, uint32_t num_cu, hipStream_t st) {
    SymHalfArgs s = sweep_args(h);
    s.steps = (h.n + 31) / 32;
    const uint32_t grid = num_cu * half_groups(KS);
    // sweeps in slices: sixteen items a workgroup at least, of 32 steps at least, and of fewer, down to two, where these leave workgroups
    // without an item.  (4096 rows are 40 items of 32 steps for 768 workgroups: 4096 x 128 in clusters, k 128, 1137 us a call
    // on two bf16 halves a value, 1349 in items of 32, 993 of 8, 762 of 4, 532 of two, 495 of one; 10,000 x 128, k 32: 529, 449, 439, 439, 435.)
    const uint64_t total = (uint64_t)s.row_tiles * s.steps / 2, least = std::min<uint64_t>(32u, std::max<uint64_t>(2u, total / grid));
    s.steps_per_slice = (uint32_t)std::min<uint64_t>(s.steps, std::max<uint64_t>(least, total / (16ull * grid)));
    s.slices = (s.steps + s.steps_per_slice - 1) / s.steps_per_slice;
    s.work_counter = h.scal + 2;
    static_assert(sizeof(SymHalfLds<KS>) <= 160 * 1024 / half_groups(KS), "so many workgroups per CU");
    GRAB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(sym_half_kernel<KS>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(SymHalfLds<KS>)));
    hipLaunchKernelGGL(sym_half_kernel<KS>, dim3(std::min(s.row_tiles * s.slices, grid)), dim3(256), sizeof(SymHalfLds<KS>), st, s);
    return GRAB_OK;
}

template <int CB, bool BOUND>
int launch_long(const SymHalfArgs& s, const uint4* columns, float* best, uint32_t num_cu, hipStream_t st) {
    constexpr size_t lds = sizeof(SymLongLds<CB, BOUND>);
    static_assert(lds + 2 * (kTileRows / 32 + CB * 2) * 2048 <= 160 * 1024, "a workgroup a CU");
    GRAB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(sym_half_long_kernel<CB, BOUND>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((sym_half_long_kernel<CB, BOUND>), dim3(std::min(s.row_tiles * s.slices, num_cu)), dim3(512), lds, st, s, columns, best);
    return GRAB_OK;
}

int launch_bounds_long(const HalfKnn& h, uint32_t num_cu, hipStream_t st) {
    SymHalfArgs s = sweep_args(h);
    s.steps = s.steps_per_slice = h.sample_places / 128;
    s.slices = 1;
    s.work_counter = h.scal + 2;
    hipLaunchKernelGGL(half_row_fragments_kernel, dim3((h.places + 255) / 256), dim3(256), 0, st, h.hn, (const float*)nullptr, s.norm_factor, h.places, h.row_frags);
    return launch_long<2, true>(s, h.sample_blocks, h.best, num_cu, st);
}

int launch_sweep_long(const HalfKnn& h, uint32_t num_cu, hipStream_t st) {
    SymHalfArgs s = sweep_args(h);
    s.steps = h.places / kTileRows;
    // twice as many slices as an XCD has under way at a time, of two tiles at least
    s.steps_per_slice = std::max(2u, (s.steps + 7u) / 8u);
    s.slices = (s.steps + s.steps_per_slice - 1) / s.steps_per_slice;
    s.work_counter = h.scal + 3;
    hipLaunchKernelGGL(half_row_fragments_kernel, dim3((h.places + 255) / 256), dim3(256), 0, st, h.hn, h.t_step, s.norm_factor, h.places, h.row_frags);
    return launch_long<4, false>(s, h.blocks, nullptr, num_cu, st);
}

}  // namespace

bool half_knn_applies(uint64_t n, uint32_t dim, int metric) {
    static_assert((1u << 23) <= kQueueColumns, "columns of the sweep");
    return n >= 4096 && n <= (1u << 23) && ((metric == kMetricL2 && dim <= 128) || dim % 32 == 0);
}

int half_knn_plan(uint32_t n, uint32_t dim, uint32_t k, int metric, HalfKnn* h) {
    h->n = n;
    h->dim = dim;
    h->ip = metric == kMetricIP;
    h->places = (n + kTileRows - 1) / kTileRows * kTileRows;
    h->n_sample = (uint32_t)std::min<size_t>(kHalfSample, n / 16);
    // The list must hold the k + 1 nearest with high probability: of them a share n_sample / n is in the sample, mean m, and
    // the rank-th nearest sample row lies beyond them all unless `rank` of them are - m + 4.5 sqrt(m) + 3 is met by some
    // one row in 10^4 (1M x 128, k 128: rank 23, 470 columns a list, 6 rows redone).
    const double m = (k + 17.0) * h->n_sample / n;
    const double rank = std::ceil(m + 4.5 * std::sqrt(m) + 3.0);
    // A list a third as long as the bound was to make it comes from a sample that does not stand for the row's surroundings.
    h->min_list = std::max(k + 1, std::min((uint32_t)(rank * n / h->n_sample / 3.0), kHalfListCap / 4));
    // of 128 classes of columns the q best stand in for that rank
    uint32_t q = 1;
    while (q < kSampleClasses / 2 && kSampleClasses * (1.0 - std::pow(1.0 - 1.0 / kSampleClasses, rank)) > q + 0.5) ++q;
    h->class_rank = q;
    h->ks = ks_of(dim);
    h->frags = dim <= 128 ? h->ks + 1 : h->ks + 2;
    h->sample_places = (h->n_sample + 127) / 128 * 128;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += (bytes + 255) & ~(size_t)255;
        return here;
    };
    h->at_blocks = take((size_t)h->places / 32 * h->frags * 1024);
    h->at_sample = take((size_t)h->sample_places / 32 * h->frags * 1024);
    h->at_row_frags = take(dim <= 128 ? 0 : (size_t)h->places / 32 * 2048);
    h->at_words = take(((size_t)h->places * 9 + h->sample_places + h->ks * 16) * 4 + kOrderBins * 4 + 64);
    h->workspace_bytes = at;
    h->id_bits = 1;
    while ((1ull << h->id_bits) < n) ++h->id_bits;
    h->list_bytes = (size_t)n * kHalfListCap * 4;
    return GRAB_OK;
}

int half_knn_lists_async(const float* data, HalfKnn* h, void* workspace, uint32_t* list, uint32_t num_cu, hipStream_t st) {
    GRAB_REQUIRE(half_knn_applies(h->n, h->dim, h->ip ? kMetricIP : kMetricL2), "internal: shape of the f16 pass");
    char* ws = static_cast<char*>(workspace);
    const uint32_t n = h->n, dim = h->dim, ks = h->ks, places = h->places;
    h->list = list;
    h->blocks = reinterpret_cast<uint4*>(ws + h->at_blocks);
    h->sample_blocks = reinterpret_cast<uint4*>(ws + h->at_sample);
    h->row_frags = reinterpret_cast<uint4*>(ws + h->at_row_frags);
    h->best = reinterpret_cast<float*>(list);  // the lists' memory, before there are lists
    static_assert(kSampleClasses <= (int)kHalfListCap, "a row's best values fit where its list will be");
    float* w = reinterpret_cast<float*>(ws + h->at_words);
    h->hn = w, w += places;
    h->cnorm = w, w += places;
    h->eps = w, w += places;
    h->bound = w, w += places;
    h->t_own = w, w += places;
    h->t_step = w, w += places;
    h->top = w, w += places;
    h->perm = reinterpret_cast<uint32_t*>(w), w += places;
    float* sample_hn = w;
    w += h->sample_places;
    // the words from here on start from zero: the lists' counts, the centre, the bins of the order, scal
    uint32_t* zeros = reinterpret_cast<uint32_t*>(w);
    h->count = zeros;
    h->centre = reinterpret_cast<float*>(zeros + places);
    h->bins = zeros + places + ks * 16;
    h->scal = h->bins + kOrderBins;
    const float nf = norm_factor(*h);
    GRAB_HIP(hipMemsetAsync(zeros, 0, ((size_t)places + ks * 16 + kOrderBins + 16) * 4, st));
    if (!h->ip) hipLaunchKernelGGL(half_centre_kernel, dim3(ks * 16), dim3(256), 0, st, data, (uint64_t)n, std::min(n, 8192u), dim, h->centre);
    hipLaunchKernelGGL(half_norms_kernel, dim3(std::min((n + 15) / 16, 2048u)), dim3(256), 0, st, data, n, dim, h->centre, h->cnorm, h->scal);
    launch_half_pack<kSpaced>(data, n, dim, ks, h->frags, nf, 1.0f, h->centre, h->cnorm, h->scal, nullptr, h->n_sample, h->sample_places, h->sample_blocks, sample_hn,
                              nullptr, st);
    launch_half_pack<kAll>(data, n, dim, ks, h->frags, nf, 1.0f, h->centre, h->cnorm, h->scal, nullptr, n, places, h->blocks, h->hn, h->eps, st);
    switch (dim <= 128 ? ks : 0u) {
        case 2: GRAB_TRY(launch_bounds_short<2>(*h, st)); break;
        case 4: GRAB_TRY(launch_bounds_short<4>(*h, st)); break;
        case 6: GRAB_TRY(launch_bounds_short<6>(*h, st)); break;
        case 8: GRAB_TRY(launch_bounds_short<8>(*h, st)); break;
        default: GRAB_TRY(launch_bounds_long(*h, num_cu, st));
    }
    hipLaunchKernelGGL(half_bound_kernel, dim3((n + 3) / 4), dim3(256), 0, st, h->best, h->hn, h->scal, n, h->class_rank, (int)h->ip, h->bound);
    // the rows once more, in descending order of their bounds
    constexpr size_t bins_lds = kOrderBins * 4;
    const uint32_t order_grid = (n + kOrderRows - 1) / kOrderRows;
    GRAB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(order_count_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bins_lds));
    GRAB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(order_place_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bins_lds));
    hipLaunchKernelGGL(order_count_kernel, dim3(order_grid), dim3(1024), bins_lds, st, h->bound, n, h->bins);
    hipLaunchKernelGGL(order_scan_kernel, dim3(1), dim3(1024), 0, st, h->bins);
    hipLaunchKernelGGL(order_place_kernel, dim3(order_grid), dim3(1024), bins_lds, st, h->bound, n, h->bins, h->perm);
    launch_half_pack<kOrdered>(data, n, dim, ks, h->frags, nf, 1.0f, h->centre, h->cnorm, h->scal, h->perm, n, places, h->blocks, h->hn, nullptr, st);
    hipLaunchKernelGGL(order_thresholds_kernel, dim3((places + 255) / 256), dim3(256), 0, st, h->bound, h->perm, h->scal, h->hn, n, places, (int)h->ip, h->t_own,
                       h->t_step, h->top);
    GRAB_HIP(hipGetLastError());
    switch (dim <= 128 ? ks : 0u) {
        case 2: GRAB_TRY(launch_sweep_short<2>(*h, num_cu, st)); break;
        case 4: GRAB_TRY(launch_sweep_short<4>(*h, num_cu, st)); break;
        case 6: GRAB_TRY(launch_sweep_short<6>(*h, num_cu, st)); break;
        case 8: GRAB_TRY(launch_sweep_short<8>(*h, num_cu, st)); break;
        default: GRAB_TRY(launch_sweep_long(*h, num_cu, st));
    }
    GRAB_HIP(hipGetLastError());
    return GRAB_OK;
}

int half_knn_finish_async(const float* data, const HalfKnn& h, uint32_t k, uint32_t redo_keep, const float* norm, const float* max_norm, uint32_t* out,
                          uint32_t* redo_count, uint32_t* redo, uint32_t* doubt, hipStream_t st) {
    FinishArgs f{};
    f.data = data;
    f.list = h.list;
    f.count = h.count;
    f.perm = h.perm;
    f.bound = h.bound;
    f.t_own = h.t_own;
    f.top = h.top;
    f.norm = norm;
    f.max_norm = max_norm;
    f.cnorm = h.cnorm;
    f.eps = h.eps;
    f.scal = h.scal;
    f.out = out;
    f.redo_count = redo_count;
    f.redo = redo;
    f.doubt = doubt;
    f.n = h.n;
    f.dim = h.dim;
    f.k = k;
    f.redo_keep = redo_keep;
    f.cap = kHalfListCap;
    f.min_list = h.min_list;
    f.id_bits = h.id_bits;
    static_assert(kHalfListCap == kFinishCap, "a list fits the wave's keys");
    if (h.ip) hipLaunchKernelGGL(knn_finish_kernel<kMetricIP>, dim3((h.n + 3) / 4), dim3(256), 0, st, f);
    else hipLaunchKernelGGL(knn_finish_kernel<kMetricL2>, dim3((h.n + 3) / 4), dim3(256), 0, st, f);
    GRAB_HIP(hipGetLastError());
    return GRAB_OK;
}

}  // namespace grab
