// Exact top-k of queries inside intervals of a row set (windows, buckets) on the f16 matrix pipe: candidates from rows rounded
// to f16 once (half_rows.hpp), scored and proven exactly like those of the kNN graph (knn_half.hip).
//
// A query is one row of the tile grid, or one per interval it admits.  Every row tile (128 rows) sweeps the union of its rows'
// columns twice: once a sample of them, one of 8 to 64 neighbours, whose values are stored and give the query a bound that a
// few hundred of its columns lie within (scan_bound_kernel), then all of them with the bound as threshold - what passes goes
// through the queue into the row's list, nothing else is ever written.  Writing the values of all columns and selecting from
// them (lists of 64 keys, k up to 16), or selecting inside the contraction with thresholds that start open (beyond), from
// rows as two bf16 halves, took for 10,000 intervals of 10,000 rows of 1M x 128 512 us of kernels at k 10 and 2.8 ms at k 40,
// for 4999 queries with 1 - 4 of 64 buckets of 200,000 x 768 540 us; this 326, 370 and 370 when it came, the first 276
// since places are reserved once an item and the bounds take what a query needs.
// What bounds it, intervals: of 178 us of sweep some 59 are matrix instructions and LDS, 50 loads of chunks, one under way at a time,
// the rest the queue (every query lists some 140 columns: a dozen in each block of 32 x 32); buckets: loads of chunks.
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

constexpr uint32_t kScanRowsTile = 128;
constexpr uint32_t kScanListCap = 2048;  // entries of a row's list
constexpr uint32_t kScanHave = 2048;     // entries of a query's lists that a wave holds,
constexpr uint32_t kScanSortCap = 1024;  // ... of which it scores and sorts the nearest
constexpr float kScanLift = 0.5f;       // the longest base row comes to [2^11, 2^12): a query may be four times as long
constexpr float kOpen = -9.0e8f;        // the threshold of a query that takes all its columns: below every value, above kNever
// A tile's queries are bounded by one of 2^shift columns each, kSampleShiftMin to kSampleShiftMax: the most that leaves a row of the
// tile's mean width 1024 values, but one of 64 at least.  The sampled columns lie apart (one_of), in blocks of their own behind
// the base's: rows that resemble their neighbours - frames of a scene, a document's passages - are sampled like any others.
// (Whole blocks of 32 adjacent columns, as it was, stand for nothing but themselves there: 2000 queries in runs of 10, 40 and 200 rows
// of 500,000 x 128, intervals of 50,000, k 10: 73, 340 and 456 queries not proven, calls of 4.2 - 4.4 ms; none and 0.24 - 0.27 now.
// The same for intervals of 1500 among those of 100,000, of which every other had no sampled block: 4.46 -> 0.64.)
constexpr uint32_t kSampleValues = 1024;
constexpr uint32_t kBoundValues = 2048;  // sampled values that a query looks at, at most: 32 a lane

// Tile-grid rows into blocks, and per query: squared norm of the rounded, scaled row (-1: not taken), what rounding moved it,
// its squared norm, its scale.  16 lanes a row.
__global__ void __launch_bounds__(256) scan_pack_kernel(const float* __restrict__ queries, const uint32_t* __restrict__ row_query, const uint32_t* __restrict__ row_lo,
                                                        const uint32_t* __restrict__ row_hi, uint32_t rows, uint32_t dim, uint32_t ks_count, uint32_t frags, int ip,
                                                        const float* __restrict__ centre, const uint32_t* __restrict__ scal, uint4* __restrict__ blocks, uint4* __restrict__ row_frags,
                                                        float* __restrict__ q_hn, float* __restrict__ q_eps, float* __restrict__ q_norm, float* __restrict__ q_scale,
                                                        uint32_t* __restrict__ flag) {
    const uint32_t p = (blockIdx.x * 256 + threadIdx.x) >> 4, j = threadIdx.x & 15;
    if (p >= rows) return;  // whole groups of 16 lanes
    const bool live = row_lo[p] < row_hi[p];
    const uint32_t q = row_query[p];
    const float4* x4 = reinterpret_cast<const float4*>(queries + (size_t)q * dim);
    const float4* c4 = reinterpret_cast<const float4*>(centre);
    float s = 0.0f;
    for (uint32_t c = j; c < (dim >> 2); c += 16) {
        const float4 v = x4[c], m = c4[c];
        const float x = v.x - m.x, y = v.y - m.y, z = v.z - m.z, w = v.w - m.w;
        s = __builtin_fmaf(x, x, __builtin_fmaf(y, y, __builtin_fmaf(z, z, __builtin_fmaf(w, w, s))));
    }
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) s += __shfl_xor(s, m, 64);
    const float scale = (ip ? scale_of(s < 3.0e38f ? s : 0.0f) : scale_of(__uint_as_float(scal[0]))) * kScanLift;
    const bool good = s < 3.0e38f && s * scale * scale < 2.68e8f;  // 2^28
    uint4* block = blocks + (size_t)(p >> 5) * frags * 64 + (p & 31);
    float sq = 0.0f, rem = 0.0f;
    for (uint32_t c = j; c < 2 * ks_count; c += 16) {
        uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            if (good && live) {
                const float4 v = x4[2 * c + h], m = c4[2 * c + h];
                const float t[4] = {v.x - m.x, v.y - m.y, v.z - m.z, v.w - m.w};
#pragma unroll
                for (uint32_t e = 0; e < 4; ++e) {
                    const float full = t[e] * scale, r = half_value(flush_half(full)), left = full - r;  // exact
                    sq = __builtin_fmaf(r, r, sq);
                    rem = __builtin_fmaf(left, left, rem);
                    w[2 * h + (e >> 1)] |= half_bits(r) << (16 * (e & 1));
                }
            }
        }
        block[(c >> 1) * 64 + (c & 1) * 32] = make_uint4(w[0], w[1], w[2], w[3]);
    }
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) {
        sq += __shfl_xor(sq, m, 64);
        rem += __shfl_xor(rem, m, 64);
    }
    if (j < 4)  // the norm's fragment, as a row has it, and zeros behind it
        row_frags[(size_t)(p >> 5) * 128 + (p & 31) + 32 * j] =
            j == 0 ? row_norm_pieces(good && live ? (ip ? 0.0f : -0.5f) * sq : kNever * kNormUnit) : make_uint4(0u, 0u, 0u, 0u);
    if (j == 0 && live) {  // (the rows of one query write the same)
        q_hn[q] = good ? sq : -1.0f;
        q_eps[q] = sqrtf(rem) / scale * 1.0001f + 1.3e-7f * sqrtf(s);
        q_norm[q] = s;
        q_scale[q] = scale;
        if (!good) *flag = 1u;
    }
}

struct ScanSweepArgs {
    const uint4* row_blocks;
    const uint4* row_frags;
    const uint4* blocks;      // base rows
    const uint32_t* items;    // [4 words]: row tile, first block, tiles of 8 blocks, block of the sample
    const uint32_t* tiles;    // [4 words] per row tile: its sample's place (of 4096 floats), blocks, first block among its shift's, shift
    const uint32_t* row_query;
    const uint32_t* row_lo;
    const uint32_t* row_hi;
    const float* q_t;
    const float* q_top;
    float* sample;
    uint32_t* list;
    uint32_t* count;
    uint32_t* work_counter;
    uint32_t n_items, frags, last_block, id_bits;
};
struct ScanTables {  // of a workgroup's 128 rows
    float t[kScanRowsTile], top[kScanRowsTile];
    uint32_t lo[kScanRowsTile], hi[kScanRowsTile];
    uint32_t block_lo[kScanRowsTile / 32], block_hi[kScanRowsTile / 32];  // what 32 rows admit between them (blocks beyond are passed over: 204 -> 198 us)
};
// What an item lists stays in LDS until the item ends: one addition in device memory then reserves the places of all its entries
// of a row, where one for every entry (1.2 million for 10,000 queries) was what the sweep waited for.  Entries that find no
// room take their own place at once.  10,000 intervals of 10,000 rows of 1M x 128: sweep 198 -> 174 us, the call 503 -> 470; 4999
// queries with 1 - 4 of 64 buckets of 200,000 x 768: 545 -> 494.
constexpr uint32_t kScanHits = 832;  // three column tiles of a row tile list some 500
struct ScanHits {
    uint32_t count[kScanRowsTile];  // of a row's entries here; then the place of the next of them in the row's list
    uint32_t entry[kScanHits];
    uint8_t row[kScanHits];
    uint32_t fill;
};
struct ScanSink {
    const ScanSweepArgs& a;
    const ScanTables& rows;
    ScanHits& hits;
    uint32_t row0 = 0, col0 = 0;  // first row and column of the item
    __device__ __forceinline__ void put(float value, uint32_t il, uint32_t col) {
        const uint32_t j = col0 + col;
        if (j < rows.lo[il] || j >= rows.hi[il]) return;  // (what a row tile sweeps, not every row of it admits)
        const float t = rows.t[il];
        const uint32_t entry = j | share_of(value + t, t, rows.top[il], a.id_bits), slot = atomicAdd(&hits.fill, 1u);
        if (slot < kScanHits) {
            hits.entry[slot] = entry;
            hits.row[slot] = (uint8_t)il;
            atomicAdd(&hits.count[il], 1u);
        } else {
            list(il, atomicAdd(&a.count[row0 + il], 1u), entry);
        }
    }
    __device__ __forceinline__ void list(uint32_t il, uint32_t at, uint32_t entry) {
        if (at < kScanListCap) a.list[(size_t)(row0 + il) * kScanListCap + at] = entry;
    }
};

// The contraction: two workgroups of four waves a CU, a tile of 128 rows x 256 columns; wave (wr, wc) owns 64 rows and 128
// columns of it.  Chunks of 32 dimensions, loads and buffers as in sym_half_long_kernel.
template <bool SAMPLE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) scan_half_kernel(const ScanSweepArgs a) {
    constexpr uint32_t kRowPart = kScanRowsTile / 32 * 128, kColPart = 8 * 128, AF = kRowPart / 256, BF = kColPart / 256;
    __shared__ v4u s_chunk0[kRowPart + kColPart], s_chunk1[kRowPart + kColPart];
    __shared__ QueueLds s_queue[SAMPLE ? 1 : 4];
    __shared__ ScanTables s_rows;
    __shared__ ScanHits s_hits;
    __shared__ uint32_t s_item;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), half = lane >> 5, l32 = lane & 31;
    const uint32_t wr = wave >> 1, wc = wave & 1, chunks = a.frags / 2, padded = (chunks + 1u) & ~1u;
    PairQueue<ScanSink> queue(ScanSink{a, s_rows, s_hits}, s_queue[SAMPLE ? 0 : wave], lane, wr * 64);
    for (;;) {
        loads_landed();   // the one too many that the item before has under way, also before the workgroup ends
        __syncthreads();  // the item before is fully drained
        if (tid == 0) s_item = atomicAdd(a.work_counter, 1u);
        __syncthreads();
        const uint32_t work = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_item);
        if (work >= a.n_items) break;  // workgroup-uniform
        const uint32_t rt = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.items[4 * work]), first = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.items[4 * work + 1]);
        const uint32_t tiles = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.items[4 * work + 2]), sampled = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.items[4 * work + 3]);
        const uint32_t row0 = rt * kScanRowsTile;
        if (!SAMPLE && tid < kScanRowsTile) {
            const uint32_t q = a.row_query[row0 + tid];
            s_hits.count[tid] = 0u;
            if (tid == 0) s_hits.fill = 0u;
            s_rows.t[tid] = a.q_t[q];
            s_rows.top[tid] = a.q_top[q];
            uint32_t lo = a.row_lo[row0 + tid], hi = a.row_hi[row0 + tid];
            s_rows.lo[tid] = lo;
            s_rows.hi[tid] = hi;
            if (lo >= hi) lo = ~0u, hi = 0u;
#pragma unroll
            for (int m = 1; m < 32; m <<= 1) {  // (waves 0 and 1, all lanes)
                lo = min(lo, (uint32_t)__shfl_xor((int)lo, m, 64));
                hi = max(hi, (uint32_t)__shfl_xor((int)hi, m, 64));
            }
            s_rows.block_lo[tid >> 5] = lo;
            s_rows.block_hi[tid >> 5] = hi;
        }
        queue.sink.row0 = row0;
        queue.sink.col0 = first * 32;
        auto load = [&](v4u* to, uint32_t tile, uint32_t c) {
            const bool norms = c + 1 >= chunks;  // workgroup-uniform
            c = min(c, chunks - 1u);
            const v4u* ra = reinterpret_cast<const v4u*>(norms ? a.row_frags : a.row_blocks);
            const uint32_t pitch = norms ? 128u : a.frags * 64, from = norms ? 0u : c * 128;
#pragma unroll
            for (uint32_t i = 0; i < AF; ++i) {
                const uint32_t at = tid + 256 * i;
                load_to_lds(ra + (size_t)(row0 / 32 + (at >> 7)) * pitch + from + (at & 127u), to + wave * 64 + 256 * i);
            }
            const v4u* rb = reinterpret_cast<const v4u*>(a.blocks) + c * 128;
#pragma unroll
            for (uint32_t i = 0; i < BF; ++i) {
                const uint32_t at = tid + 256 * i, block = min(first + 8 * tile + (at >> 7), a.last_block);  // (the base's last block is padding)
                load_to_lds(rb + (size_t)block * a.frags * 64 + (at & 127u), to + kRowPart + wave * 64 + 256 * i);
            }
        };
        uint32_t tile = 0, c = 0, tile_next = 0, c_next = 0;  // what is multiplied, and what was asked for last
        auto advance = [&]() {
            if (++c_next == padded) {
                if (tile_next + 1 < tiles) {
                    ++tile_next;
                    c_next = 0;
                } else {
                    c_next = padded - 1;
                }
            }
        };
        v16f acc[2][4];
        auto multiply = [&](const v4u* from, auto first_chunk) {
            constexpr bool FIRST = decltype(first_chunk)::value;
            const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t ks = 0; ks < 2; ++ks) {
                v8h x[2], y[4];
#pragma unroll
                for (uint32_t rb = 0; rb < 2; ++rb) x[rb] = __builtin_bit_cast(v8h, from[(wr * 2 + rb) * 128 + ks * 64 + lane]);
#pragma unroll
                for (uint32_t cb = 0; cb < 4; ++cb) y[cb] = __builtin_bit_cast(v8h, from[kRowPart + (wc * 4 + cb) * 128 + ks * 64 + lane]);
#pragma unroll
                for (uint32_t cb = 0; cb < 4; ++cb)
#pragma unroll
                    for (uint32_t rb = 0; rb < 2; ++rb)
                        acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[rb], y[cb], FIRST && ks == 0 ? zero : acc[rb][cb], 0, 0, 0);
            }
        };
        load(s_chunk0, 0, 0);
        loads_landed();
        __syncthreads();  // first chunk and row tables visible
        uint32_t from[2], to[2];  // the first column of a block that the wave's row blocks take, and the first beyond
#pragma unroll
        for (uint32_t rb = 0; rb < 2 && !SAMPLE; ++rb) {
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_rows.block_lo[wr * 2 + rb]);
            from[rb] = lo & ~31u;
            to[rb] = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_rows.block_hi[wr * 2 + rb]);
        }
        for (;;) {
            advance();
            load(s_chunk1, tile_next, c_next);
            if (c == 0) multiply(s_chunk0, std::true_type{});
            else multiply(s_chunk0, std::false_type{});
            loads_landed();
            __syncthreads();  // everyone is through with this chunk, the next one is there
            advance();
            load(s_chunk0, tile_next, c_next);
            if (c + 1 < chunks) multiply(s_chunk1, std::false_type{});
            c += 2;
            if (c == padded) {
#pragma unroll
                for (uint32_t cb = 0; cb < 4; ++cb) {
                    const uint32_t nth = 8 * tile + wc * 4 + cb;
                    if (SAMPLE) {
                        const uint32_t* t = a.tiles + 4 * rt;
                        const uint32_t pitch = t[1] * 32, at = (sampled + nth) * 32 + l32;
                        float* out = a.sample + (size_t)t[0] * 4096 + (size_t)(wr * 64 + 4 * half) * pitch + at;
#pragma unroll
                        for (uint32_t rb = 0; rb < 2; ++rb)  // (the rows one after the other: 32 addresses at once do not fit the registers)
#pragma unroll
                            for (uint32_t v = 0; v < 16; ++v) {
                                *out = acc[rb][cb][v];
                                out += (size_t)pitch * (v % 4 == 3 ? 5 : 1);
                            }
                    } else {
                        const uint32_t j0 = min(first + nth, a.last_block) * 32;
#pragma unroll
                        for (uint32_t rb = 0; rb < 2; ++rb)  // what passes here and no row admits would fall in put()
                            if (j0 >= from[rb] && j0 < to[rb]) queue.offer(acc[rb][cb], j0 - first * 32 + l32, rb);  // (row numbers go up to 2^31)
                    }
                }
                if (++tile == tiles) break;  // workgroup-uniform
                c = 0;
            }
            loads_landed();
            __syncthreads();
        }
        if (!SAMPLE) {
            queue.finish();
            __syncthreads();
            if (tid < kScanRowsTile && s_hits.count[tid] != 0u) s_hits.count[tid] = atomicAdd(&a.count[row0 + tid], s_hits.count[tid]);
            __syncthreads();
            for (uint32_t i = tid, n = min(s_hits.fill, kScanHits); i < n; i += 256) {
                const uint32_t il = s_hits.row[i];
                queue.sink.list(il, atomicAdd(&s_hits.count[il], 1u), s_hits.entry[i]);
            }
        }
    }
}

// A query's rows as scan_bound_kernel's lanes hold them, a row a lane: place of the row's sampled values, the interval, the shift,
// the tile's first sampled value and the interval's; n values are looked at, as the at-th and those after it of all that are.
struct SampledRow {
    uint32_t row = 0, lo = 0, hi = 0, shift = kSampleShiftMin, first = 0, s0 = 0, place = 0, pitch = 0, n = 0, at = 0;
};
__device__ __forceinline__ uint32_t lane_value(uint32_t v, uint32_t lane) {  // `lane` the same for the whole wave
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}
// The threshold that about `want` of the query's columns reach; kOpen: take them all.  PER values a lane, requested together.  ONE:
// the query has one row.  (With 32 values a lane and any number of rows for every query, most of the kernel was instructions
// on values that are not there: 10,000 intervals 53 -> 33 us, 10,000 queries with 1 - 4 buckets of 1M x 768 152 -> 119.)
template <int PER, bool ONE>
__device__ __forceinline__ float scan_threshold(const float* __restrict__ sample, const SampledRow& mine, uint32_t lane, uint32_t nl, uint32_t every, uint32_t n_all,
                                                uint32_t columns, uint32_t k, uint32_t num_base) {
    const uint32_t rows = ONE ? 1u : nl;
    float v[PER], w[ONE ? 1 : PER];
    uint32_t of[ONE ? 1 : PER];  // the row, or none
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        v[i] = -__builtin_inff();  // (a value that is there is finite)
        if (!ONE) {
            w[i] = 0.0f;
            of[i] = 0xFFu;
        }
    }
    uint32_t inside_one = 0;
    for (uint32_t r = 0; r < rows; ++r) {
        const uint32_t rr = lane_value(mine.row, r), rlo = lane_value(mine.lo, r), rhi = lane_value(mine.hi, r), shift = lane_value(mine.shift, r);
        const uint32_t s0 = lane_value(mine.s0, r), from = s0 - lane_value(mine.first, r), rn = lane_value(mine.n, r), rat = lane_value(mine.at, r);
        const float* src = sample + (size_t)lane_value(mine.place, r) * 4096 + (size_t)(rr % kScanRowsTile) * lane_value(mine.pitch, r);
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            if (64 * i < rat + rn && 64 * i + 64 > rat) {  // wave-uniform
                const uint32_t g = 64 * i + lane - rat, col = one_of(s0 + g * every, shift, num_base);
                const bool in = g < rn && col >= rlo && col < rhi;  // (g wraps round before the row's first value)
                if (in) {
                    v[i] = src[from + g * every];
                    if (!ONE) of[i] = r;
                }
                if (ONE) inside_one += (uint32_t)__popcll(__ballot(in));
            }
        }
    }
    float weight_max = 0.0f;
    for (uint32_t r = 0; r < rows; ++r) {
        uint32_t inside = inside_one;
        if (!ONE) {
#pragma unroll
            for (uint32_t i = 0; i < PER; ++i)
                if (64 * i < n_all) inside += (uint32_t)__popcll(__ballot(of[i] == r));
        }
        const float weight = inside ? (float)(lane_value(mine.hi, r) - lane_value(mine.lo, r)) / (float)inside : 0.0f;
        weight_max = fmaxf(weight_max, weight);
        if (!ONE) {
#pragma unroll
            for (uint32_t i = 0; i < PER; ++i) w[i] = of[i] == r ? weight : w[i];
        }
    }
    const float m = (float)k + 9.0f, want = fminf(m + 4.5f * sqrtf(m * weight_max) + 2.0f * weight_max, 800.0f);
    if ((float)columns <= 1.3f * want && columns <= kScanSortCap) return kOpen;
    auto reach = [&](float t) {  // columns that reach t
        if (ONE) {
            uint32_t n = 0;
#pragma unroll
            for (uint32_t i = 0; i < PER; ++i)
                if (64 * i < n_all) n += (uint32_t)__popcll(__ballot(v[i] >= t));
            return (float)n * weight_max;
        }
        float c = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i)
            if (64 * i < n_all) c += v[i] >= t ? w[ONE ? 0 : i] : 0.0f;
#pragma unroll
        for (int x = 1; x < 64; x <<= 1) c += __shfl_xor(c, x, 64);
        return c;
    };
    float high = -__builtin_inff(), low = __builtin_inff();
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        high = fmaxf(high, v[i]);
        low = fminf(low, v[i] > -__builtin_inff() ? v[i] : __builtin_inff());
    }
#pragma unroll
    for (int x = 1; x < 64; x <<= 1) {
        high = fmaxf(high, __shfl_xor(high, x, 64));
        low = fminf(low, __shfl_xor(low, x, 64));
    }
    if (!(low < high && reach(low) >= want)) return kOpen;
    for (int it = 0; it < 20; ++it) {
        const float mid = 0.5f * (low + high), c = reach(mid);
        if (c >= want) {
            low = mid;
            if (c < 1.08f * want || (ONE && c - weight_max < want)) break;  // (one value less would not do)
        } else {
            high = mid;
        }
    }
    return fmaxf(low, kOpen);
}

// One wave per query: the threshold.  Each row's sampled columns stand for its columns, a value for as many (its weight) as the
// sampling skipped; the threshold is the value that about `want` columns reach: so many that the k nearest are among them but
// for one query in 10^7 - of k columns a sample holds k / weight, give or take the root of that - and what the list's last
// column needs to be beyond the k-th by.  A query with few columns takes all.
__global__ void __launch_bounds__(256) scan_bound_kernel(const float* __restrict__ sample, const uint32_t* __restrict__ tiles, const uint32_t* __restrict__ row_lo,
                                                         const uint32_t* __restrict__ row_hi, const uint32_t* __restrict__ list_off, const uint32_t* __restrict__ lists,
                                                         const float* __restrict__ q_hn, uint32_t nq, uint32_t k, int ip, uint32_t num_base, float* __restrict__ q_t,
                                                         float* __restrict__ q_top, uint4* __restrict__ row_frags) {
    const uint32_t lane = threadIdx.x & 63, q = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (q >= nq) return;  // whole waves
    const uint32_t l0 = list_off[q], nl = list_off[q + 1] - l0;  // at most 64 rows
    if (nl == 0) return;
    // lane r: row r's interval, and which of its tile's sampled columns stand for it
    SampledRow mine;
    uint32_t sampled = 0;
    if (lane < nl) {
        mine.row = lists[l0 + lane];
        mine.lo = row_lo[mine.row];
        mine.hi = row_hi[mine.row];
        const uint32_t* t = tiles + 4 * (mine.row / kScanRowsTile);
        mine.place = t[0], mine.pitch = t[1] * 32, mine.first = t[2] * 32, mine.shift = t[3];
        mine.s0 = mine.lo >> mine.shift;
        sampled = ((mine.hi - 1) >> mine.shift) + 1 - mine.s0;  // (no row of a list is empty)
    }
    auto wave_sum = [&](uint32_t v) {  // (zero in the lanes that hold no row)
        if (nl == 1) return lane_value(v, 0);
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) v += __shfl_xor(v, m, 64);
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
    };
    const uint32_t columns = wave_sum(mine.hi - mine.lo), all = wave_sum(sampled);
    const float hn = q_hn[q], top = ip ? sqrtf(fmaxf(hn, 0.0f)) * 4096.0f : 0.0f;
    float t_out = kOpen;
    if (columns > 256) {
        const uint32_t every = (all + kBoundValues - 65 - 1) / (kBoundValues - 65);  // one value in so many is looked at
        mine.n = (sampled + every - 1) / every;
        for (uint32_t r = 0; r + 1 < nl; ++r) {
            const uint32_t n_r = lane_value(mine.n, r);
            if (lane > r) mine.at += n_r;
        }
        const uint32_t n_all = wave_sum(mine.n);
        if (nl == 1 && n_all <= kBoundValues / 2) t_out = scan_threshold<kBoundValues / 128, true>(sample, mine, lane, nl, every, n_all, columns, k, num_base);
        else if (nl == 1) t_out = scan_threshold<kBoundValues / 64, true>(sample, mine, lane, nl, every, n_all, columns, k, num_base);
        else if (n_all <= kBoundValues / 2) t_out = scan_threshold<kBoundValues / 128, false>(sample, mine, lane, nl, every, n_all, columns, k, num_base);
        else t_out = scan_threshold<kBoundValues / 64, false>(sample, mine, lane, nl, every, n_all, columns, k, num_base);
    }
    if (lane == 0) {
        q_t[q] = t_out;
        q_top[q] = top;
    }
    // the query's rows carry the threshold from here on (one that is not taken never passes)
    if (lane < nl && hn >= 0.0f) row_frags[(size_t)(mine.row >> 5) * 128 + (mine.row & 31)] = row_norm_pieces((ip ? 0.0f : -0.5f) * hn - t_out);
}

// One wave per query: the lists of its rows - one threshold, so their entries compare - to results, as knn_finish_kernel does it
struct ScanFinishArgs {
    HalfScanArgs a;
    const uint32_t* list;
    const uint32_t* count;
    const float* q_t;
    const float* q_top;
    const float* q_eps;
    const float* q_norm;
    const float* q_scale;
    const uint32_t* scal;
    uint32_t nq, k, dim, id_bits;
};
template <int METRIC>
__global__ void __launch_bounds__(256) scan_finish_kernel(const ScanFinishArgs f) {
    __shared__ uint64_t keys_all[4][kScanSortCap];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t q = blockIdx.x * 4 + wave;
    if (q >= f.nq) return;  // wave-uniform; no barrier below
    uint64_t* keys = keys_all[wave];
    static_assert(kScanHave * 4 <= kScanSortCap * 8, "entries, then keys, in the same place");
    uint32_t* ents = reinterpret_cast<uint32_t*>(keys);
    const uint32_t l0 = f.a.list_off[q], l1 = f.a.list_off[q + 1];
    const uint32_t id_mask = (1u << f.id_bits) - 1u, parts = 1u << (32u - f.id_bits), need = f.k - 1;
    uint32_t total = 0;
    bool whole = true;
    for (uint32_t l = l0; l < l1; ++l) {
        const uint32_t c = f.count[f.a.lists[l]];
        whole = whole && c <= kScanListCap;
        total += whole ? c : 0u;
    }
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto up_to = [&](uint32_t last) {  // entries of all lists up to `last` into LDS: how many
        uint32_t n = 0;
        for (uint32_t l = l0; l < l1; ++l) {
            const uint32_t row = f.a.lists[l], c = f.count[row];
            for (uint32_t g0 = 0; g0 < c; g0 += 64) {
                const uint32_t e = g0 + lane < c ? f.list[(size_t)row * kScanListCap + g0 + lane] : 0u;
                const bool in = g0 + lane < c && e <= last;
                const uint64_t b = __ballot(in);
                if (in) ents[n + (uint32_t)__popcll(b & ((1ull << lane) - 1ull))] = e;
                n += (uint32_t)__popcll(b);
            }
        }
        return n;
    };
    // More entries than a wave holds (many rows, a coarse sample): the nearest parts of them, as many as fit.  Counted in 1024 bins,
    // one pass over the lists; halving the parts with a pass each took 20 (a query of 52 pieces of 3M rows x 128: 507 us the call, now 343;
    // rows as two bf16 halves 369.  From 1024 entries on, which it scores, and not from the 2048 it holds: one of 25 pieces 290 us, now
    // 204; halves 250).
    uint32_t kept_part = parts - 1u;
    if (whole && total > kScanHave) {
        constexpr uint32_t kBins = 1024;
        const uint32_t shift = max(f.id_bits, 22u);  // an entry's bin: its part, or the upper ten bits of it
        for (uint32_t g = lane; g < kBins; g += 64) ents[g] = 0u;
        wave_sync();
        for (uint32_t l = l0; l < l1; ++l) {
            const uint32_t row = f.a.lists[l], c = f.count[row];
            for (uint32_t g = lane; g < c; g += 64) atomicAdd(&ents[f.list[(size_t)row * kScanListCap + g] >> shift], 1u);
        }
        wave_sync();
        uint32_t bins[kBins / 64], sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < kBins / 64; ++i) sum += bins[i] = ents[lane * (kBins / 64) + i];
        uint32_t upto = sum;  // ... of this lane's bins and those before
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const uint32_t before = __shfl_up(upto, m, 64);
            upto += lane >= m ? before : 0u;
        }
        uint32_t fit = 0, at = upto - sum;  // this lane's bins that fit; those of the lanes before do where one of these does
#pragma unroll
        for (uint32_t i = 0; i < kBins / 64; ++i) {
            at += bins[i];
            fit += at <= kScanHave ? 1u : 0u;
        }
#pragma unroll
        for (int m = 32; m > 0; m >>= 1) fit += __shfl_xor(fit, m, 64);
        whole = fit != 0;
        kept_part = (uint32_t)((((uint64_t)fit << shift) - 1u) >> f.id_bits);
        wave_sync();
    }
    uint32_t have = whole ? up_to((kept_part << f.id_bits) | id_mask) : 0u;
    const float t = l1 > l0 ? f.q_t[q] : kOpen;
    const bool open = t <= kOpen;  // all columns are in the lists
    if (!whole || (!open && have <= need) || (open && kept_part != parts - 1u)) {
        if (lane == 0) f.a.doubt[1 + atomicAdd(f.a.doubt, 1u)] = q;
        return;
    }
    wave_sync();
    // 1024 of them go to registers; more, which is rare, stay in LDS until it is known which few can matter (registers for 2048: 37 ->
    // 44 us for 10,000 intervals of 10,000 rows of 1M x 128)
    constexpr int kEnts = kScanSortCap / 64;
    uint32_t ent[kEnts];
    const bool many = have > kScanSortCap;
#pragma unroll
    for (int i = 0; i < kEnts; ++i) ent[i] = !many && (uint32_t)(i * 64 + lane) < have ? ents[i * 64 + lane] : kInvalidId;
    __builtin_amdgcn_wave_barrier();
    uint32_t last_part = parts - 1u;
    double bound = 0.0, form = 0.0, e_far = 0.0;
    const double u = 5.9604644775390625e-08, dim = f.dim, rescore = (f.dim / 8 + 8) * u;
    auto within = [&](uint32_t part) {  // entries in the parts up to `part`
        uint32_t c = 0;
        const uint32_t last = (part << f.id_bits) | id_mask;
        if (many) {
            for (uint32_t g = 0; g < have; g += 64) c += (uint32_t)__popcll(__ballot(g + lane < have && ents[g + lane] <= last));
            return c;
        }
#pragma unroll
        for (int i = 0; i < kEnts; ++i)
            if ((uint32_t)(i * 64) < have) c += (uint32_t)__popcll(__ballot((uint32_t)(i * 64 + lane) < have && ent[i] <= last));
        return c;
    };
    if (!open) {
        uint32_t low = 0, high = parts - 1u, n_high = have;
        while (low < high && n_high > need + 2) {
            const uint32_t mid = (low + high) >> 1, c = within(mid);
            if (c > need) {
                high = mid;
                n_high = c;
            } else {
                low = mid + 1;
            }
        }
        const double eps = f.q_eps[q], eps_max = __uint_as_float(f.scal[1]), cn = f.q_norm[q], cn_max = __uint_as_float(f.scal[0]);
        const double base_scale = (double)scale_of(__uint_as_float(f.scal[0])) * kScanLift, unit = (METRIC == kMetricL2 ? -2.0 : -1.0) / (base_scale * (double)f.q_scale[q]);
        // (the error of the products formed here, and none of a form on the rows as they are: with rows far from the origin, where that
        // one tells nothing apart, these are centred.  100,000 x 128 about 100 in every coordinate, 300 windows of 20,000: 226 not proven
        // and 3443 us a call with both, 155 with rows as two bf16 halves)
        if (METRIC == kMetricL2) {
            form = (3.25 * dim + 96.0) * u * (cn + cn_max);
            e_far = eps + eps_max;
        } else {
            form = (2.0 * dim + 96.0) * u * sqrt(cn * cn_max);
            e_far = eps * sqrt(cn_max) + (sqrt(cn) + eps) * eps_max + form;
        }
        const double top = f.q_top[q], way = top - (double)t, edge = (top - way * (high + 2.0) / parts) * unit;
        bound = (double)t * unit;
        double cutoff;
        if (METRIC == kMetricL2) {
            const double r = sqrt(edge + form) * (1.0 + 2.0 * rescore) + 2.0 * e_far;
            cutoff = r * r + form;
        } else {
            cutoff = edge + 2.0 * e_far + 2.0 * form;
        }
        const double far_part = (top - cutoff / unit) / way * parts + 1.0;
        last_part = far_part < (double)(parts - 1u) ? (uint32_t)fmax(far_part, 0.0) : parts - 1u;  // (all of them where it is not a number)
    }
    if (many) {
        if (within(last_part) > kScanSortCap) {
            if (lane == 0) f.a.doubt[1 + atomicAdd(f.a.doubt, 1u)] = q;
            return;
        }
        uint32_t kept = 0;  // those up to last_part to the front: a place is read before anything is written there
        for (uint32_t g = 0; g < have; g += 64) {
            const uint32_t e = g + lane < have ? ents[g + lane] : kInvalidId;
            const bool in = g + lane < have && e <= ((last_part << f.id_bits) | id_mask);
            const uint64_t b = __ballot(in);
            wave_sync();
            if (in) ents[kept + (uint32_t)__popcll(b & ((1ull << lane) - 1ull))] = e;
            kept += (uint32_t)__popcll(b);
        }
        wave_sync();
        have = kept;
#pragma unroll
        for (int i = 0; i < kEnts; ++i) ent[i] = (uint32_t)(i * 64 + lane) < have ? ents[i * 64 + lane] : kInvalidId;
        __builtin_amdgcn_wave_barrier();
    }
    uint32_t n_score = 0;
    {
        const uint32_t last = (last_part << f.id_bits) | id_mask;
#pragma unroll
        for (int i = 0; i < kEnts; ++i) {
            if ((uint32_t)(i * 64) < have) {
                const bool in = (uint32_t)(i * 64 + lane) < have && ent[i] <= last;
                const uint64_t b = __ballot(in);
                if (in) keys[n_score + (uint32_t)__popcll(b & ((1ull << lane) - 1ull))] = ent[i] & id_mask;
                n_score += (uint32_t)__popcll(b);
            }
        }
    }
    wave_sync();
    const float4* q4 = reinterpret_cast<const float4*>(f.a.queries + (size_t)q * f.dim);
    const int grp = lane >> 3, j = lane & 7;
    for (uint32_t c0 = 0; c0 < n_score; c0 += 16) {
        const uint32_t ca = c0 + grp, cb = ca + 8;
        if (ca >= n_score) continue;
        const uint32_t ia = (uint32_t)keys[ca], ib = cb < n_score ? (uint32_t)keys[cb] : ia;
        float da = 0.0f, db = 0.0f;
        fold_rows_any<METRIC, true>(reinterpret_cast<const float4*>(f.a.data + (size_t)ia * f.dim), reinterpret_cast<const float4*>(f.a.data + (size_t)ib * f.dim), q4, j,
                                    f.dim >> 2, da, db);
        da = group8_sum(da);
        db = group8_sum(db);
        if (j == 0) keys[ca] = make_sel_key(METRIC == kMetricIP ? -da : da, ia);
        if (j == 0 && cb < n_score) keys[cb] = make_sel_key(METRIC == kMetricIP ? -db : db, ib);
    }
    wave_sync();
    auto sorted = [&](auto per_lane) {
        constexpr int NPL = decltype(per_lane)::value;
        uint64_t x[NPL];
#pragma unroll
        for (int i = 0; i < NPL; ++i) x[i] = (uint32_t)(lane * NPL + i) < n_score ? keys[lane * NPL + i] : kInvalidKey;
        wave_bitonic_sort<NPL>(x);
#pragma unroll
        for (int i = 0; i < NPL; ++i) keys[lane * NPL + i] = x[i];
    };
    if (n_score <= 64) sorted(std::integral_constant<int, 1>{});
    else if (n_score <= 256) sorted(std::integral_constant<int, 4>{});
    else sorted(std::integral_constant<int, 16>{});
    wave_sync();
    if (!open) {  // every column of the query that is in no list lies at or beyond the bound
        const double last = (double)ord_float((uint32_t)(keys[need] >> 32));
        bool proven;
        if (METRIC == kMetricL2) {
            const double near_b = sqrt(fmax(bound - form, 0.0)) - e_far, out = near_b > 0.0 ? near_b * near_b : 0.0;
            proven = last < out - rescore * out;
        } else {
            proven = last < bound - e_far - form;
        }
        if (!proven || last_part > kept_part) {  // (also where something is not a number)
            if (lane == 0) f.a.doubt[1 + atomicAdd(f.a.doubt, 1u)] = q;
            return;
        }
    }
    for (uint32_t o = lane; o < f.k; o += 64) {
        const uint64_t key = o < n_score ? keys[o] : kInvalidKey;
        const bool valid = key != kInvalidKey;
        f.a.out_ids[(size_t)q * f.k + o] = valid ? (int64_t)(key & 0xFFFFFFFFull) : -1;
        f.a.out_dist[(size_t)q * f.k + o] = valid ? ord_float((uint32_t)(key >> 32)) : kDistMax;
    }
}

size_t base_places(size_t n) { return (n + 255) / 256 * 256 + 256; }  // a block of padding at least, which stands for every block past the end

}  // namespace

bool half_scan_takes(uint64_t widest) { return widest <= (uint64_t)(kBoundValues - 65) << kSampleShiftMax; }

size_t sample_places(size_t n, uint32_t shift) { return (((n - 1) >> shift) + 32) / 32 * 32; }

size_t half_base_bytes(size_t n, uint32_t dim) {
    size_t places = base_places(n);
    for (uint32_t shift = kSampleShiftMin; shift <= kSampleShiftMax; ++shift) places += sample_places(n, shift);
    return places / 32 * (dim / 16 + 2) * 1024 + base_places(n) * 4 + n * 8 + (size_t)dim * 4 + 16 * 4 + 1024;
}

int half_base_async(const float* data, size_t n, uint32_t dim, int metric, void* mem, HalfBase* out, hipStream_t st) {
    GRAB_REQUIRE(dim % 32 == 0 && n < (1ull << 31), "internal: base rows of the f16 scans");
    HalfBase& b = *out;
    b.n = (uint32_t)n;
    b.dim = dim;
    b.ks = dim / 16;
    b.frags = b.ks + 2;
    b.ip = metric == kMetricIP;
    const uint32_t places = (uint32_t)base_places(n);
    b.last_block = places / 32 - 1;
    char* m = static_cast<char*>(mem);
    auto take = [&](size_t bytes) {
        char* here = m;
        m += (bytes + 255) & ~(size_t)255;
        return here;
    };
    uint32_t blocks = places / 32;
    for (uint32_t shift = kSampleShiftMin; shift <= kSampleShiftMax; ++shift) {
        b.sample_first[shift] = blocks;
        blocks += (uint32_t)sample_places(n, shift) / 32;
    }
    b.last_sample_block = blocks - 1;
    b.blocks = reinterpret_cast<uint4*>(take((size_t)blocks * b.frags * 1024));
    b.centre = reinterpret_cast<float*>(take((size_t)dim * 4 + 64));
    b.scal = reinterpret_cast<uint32_t*>(b.centre + dim);
    float* hn = reinterpret_cast<float*>(take((size_t)places * 4));
    float* cnorm = reinterpret_cast<float*>(m);
    float* eps = cnorm + n;
    GRAB_HIP(hipMemsetAsync(b.centre, 0, (size_t)dim * 4 + 64, st));
    if (b.ip) launch_one_way(data, n, dim, reinterpret_cast<float*>(b.blocks), b.scal + kScalOneWay, st);  // (before there are blocks)
    else hipLaunchKernelGGL(half_centre_kernel, dim3(dim), dim3(256), 0, st, data, (uint64_t)n, (uint32_t)std::min<size_t>(n, 8192), dim, b.centre);
    hipLaunchKernelGGL(half_norms_kernel, dim3((uint32_t)std::min<size_t>((n + 15) / 16, 2048)), dim3(256), 0, st, data, b.n, dim, b.centre, cnorm, b.scal);
    launch_half_pack<kAll>(data, n, dim, b.ks, b.frags, b.ip ? 0.0f : -0.5f, kScanLift, b.centre, cnorm, b.scal, nullptr, b.n, places, b.blocks, hn, eps, st);
    for (uint32_t shift = kSampleShiftMin; shift <= kSampleShiftMax; ++shift)  // (their norms go where the rows' own were, which nothing reads)
        launch_half_pack<kOneOf>(data, n, dim, b.ks, b.frags, b.ip ? 0.0f : -0.5f, kScanLift, b.centre, cnorm, b.scal, nullptr, shift, (uint32_t)sample_places(n, shift),
                                 b.blocks + (size_t)b.sample_first[shift] * b.frags * 64, hn, nullptr, st);
    GRAB_HIP(hipGetLastError());
    return GRAB_OK;
}

bool half_scan_plan(const HalfBase& b, uint32_t num_cu, const uint32_t* h_row_lo, const uint32_t* h_row_hi, size_t max_bytes, HalfScan* s) {
    const uint32_t row_tiles = s->rows / kScanRowsTile;
    // tiles of 8 blocks, 256 columns; an item is as many as leave every workgroup some four of them
    constexpr uint32_t kItemTiles = 32;  // ... at most
    static_assert(kItemTiles * 256 <= kQueueColumns, "columns of an item");
    uint64_t total = 0;
    for (uint32_t t = 0; t < row_tiles; ++t) total += (s->tile_hi[t] - s->tile_lo[t] + 1) / 2;
    const uint32_t per = (uint32_t)std::min<uint64_t>(kItemTiles, std::max<uint64_t>(1, total / (2ull * num_cu * 4)));
    auto blocks_of = [&](uint32_t t) { return 4u * (s->tile_hi[t] - s->tile_lo[t]); };
    struct Sampled {
        uint32_t shift, first, blocks;  // first block among the shift's, blocks in whole tiles
    };
    std::vector<Sampled> samples(row_tiles);
    uint64_t sampled = 0;
    size_t n_sweep = 0;
    for (uint32_t t = 0; t < row_tiles; ++t) {
        uint64_t width = 0;
        uint32_t live = 0;
        for (uint32_t r = t * kScanRowsTile; r < (t + 1) * kScanRowsTile; ++r) {
            width += h_row_hi[r] - h_row_lo[r];  // (never the other way round)
            live += h_row_hi[r] > h_row_lo[r] ? 1u : 0u;
        }
        Sampled& x = samples[t];
        x.shift = kSampleShiftMin;
        while (x.shift < kSampleShiftMax && (width >> x.shift) > (uint64_t)live * kSampleValues) ++x.shift;
        x.first = (s->tile_lo[t] * 128u >> x.shift) / 32;
        x.blocks = (((s->tile_hi[t] * 128u - 1u) >> x.shift) / 32 - x.first + 8) / 8 * 8;
        sampled += x.blocks;
        n_sweep += ((blocks_of(t) + 7) / 8 + per - 1) / per;
    }
    if (sampled * 4096 * 4 + (size_t)s->rows * kScanListCap * 4 > max_bytes) return false;
    const size_t n_sample = sampled / 8;
    s->at_tiles = 0;
    s->at_sweep = (size_t)row_tiles * 4;
    s->at_sample = s->at_sweep + n_sweep * 4;
    s->words.resize(s->at_sample + n_sample * 4);
    uint32_t *tile = s->words.data(), *sweep = tile + s->at_sweep, *sample = tile + s->at_sample;
    uint32_t at = 0;
    auto put = [](uint32_t*& to, uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
        to[0] = a, to[1] = b, to[2] = c, to[3] = d;
        to += 4;
    };
    for (uint32_t t = 0; t < row_tiles; ++t) {
        const uint32_t first = 4 * s->tile_lo[t], blocks = blocks_of(t);
        const Sampled& x = samples[t];
        for (uint32_t done = 0; done < blocks; done += 8 * per) put(sweep, t, first + done, std::min(per, (blocks - done + 7) / 8), 0u);
        for (uint32_t i = 0; i < x.blocks; i += 8) put(sample, t, b.sample_first[x.shift] + x.first + i, 1u, i);
        put(tile, at, x.blocks, x.first, x.shift);  // a row tile's sample: 128 rows of 32 floats a block
        at += x.blocks;
    }
    s->sweep_items = (uint32_t)n_sweep;
    s->sample_items = (uint32_t)n_sample;
    s->sample_floats = (size_t)at * 4096;
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    s->workspace_bytes = up((size_t)s->rows / 32 * b.frags * 1024) + up((size_t)s->rows / 32 * 2048) + up(s->sample_floats * 4) + up((size_t)s->rows * kScanListCap * 4) +
                         up((size_t)s->nq * 24) + up((size_t)s->rows * 4 + 64 + (size_t)s->nq * 4);
    return s->workspace_bytes <= max_bytes;
}

int half_scan_async(const HalfBase& b, const HalfScan& s, const HalfScanArgs& given, void* workspace, uint32_t num_cu, uint32_t** left, hipStream_t st) {
    HalfScanArgs a = given;
    char* m = static_cast<char*>(workspace);
    auto take = [&](size_t bytes) {
        char* here = m;
        m += (bytes + 255) & ~(size_t)255;
        return here;
    };
    const uint32_t rows = s.rows, nq = s.nq;
    ScanSweepArgs w{};
    uint4* row_blocks = reinterpret_cast<uint4*>(take((size_t)rows / 32 * b.frags * 1024));
    uint4* row_frags = reinterpret_cast<uint4*>(take((size_t)rows / 32 * 2048));
    w.sample = reinterpret_cast<float*>(take(s.sample_floats * 4));
    w.list = reinterpret_cast<uint32_t*>(take((size_t)rows * kScanListCap * 4));
    float* q_hn = reinterpret_cast<float*>(take((size_t)nq * 24));
    float *q_eps = q_hn + nq, *q_norm = q_eps + nq, *q_scale = q_norm + nq, *q_t = q_scale + nq, *q_top = q_t + nq;
    // from zero: the lists' counts, two work counters, whether a query is not taken, the queries not proven; then which these are
    w.count = reinterpret_cast<uint32_t*>(take((size_t)rows * 4 + 64 + (size_t)nq * 4));
    uint32_t* counters = w.count + rows;
    a.flag = *left = counters + 2;
    a.doubt = counters + 3;
    GRAB_HIP(hipMemsetAsync(w.count, 0, (size_t)rows * 4 + 64, st));
    hipLaunchKernelGGL(scan_pack_kernel, dim3(rows / 16), dim3(256), 0, st, a.queries, a.row_query, a.row_lo, a.row_hi, rows, b.dim, b.ks, b.frags, (int)b.ip, b.centre, b.scal,
                       row_blocks, row_frags, q_hn, q_eps, q_norm, q_scale, a.flag);
    w.row_blocks = row_blocks;
    w.row_frags = row_frags;
    w.blocks = b.blocks;
    w.tiles = a.words + s.at_tiles;
    w.row_query = a.row_query;
    w.row_lo = a.row_lo;
    w.row_hi = a.row_hi;
    w.q_t = q_t;
    w.q_top = q_top;
    w.frags = b.frags;
    w.last_block = b.last_sample_block;
    w.id_bits = 1;
    while ((1ull << w.id_bits) < b.n) ++w.id_bits;
    w.items = a.words + s.at_sample;
    w.n_items = s.sample_items;
    w.work_counter = counters;
    hipLaunchKernelGGL(scan_half_kernel<true>, dim3(std::min(s.sample_items, 2 * num_cu)), dim3(256), 0, st, w);
    hipLaunchKernelGGL(scan_bound_kernel, dim3((nq + 3) / 4), dim3(256), 0, st, w.sample, w.tiles, a.row_lo, a.row_hi, a.list_off, a.lists, q_hn, nq, s.k, (int)b.ip, b.n, q_t, q_top,
                       row_frags);
    w.last_block = b.last_block;
    w.items = a.words + s.at_sweep;
    w.n_items = s.sweep_items;
    w.work_counter = counters + 1;
    hipLaunchKernelGGL(scan_half_kernel<false>, dim3(std::min(s.sweep_items, 2 * num_cu)), dim3(256), 0, st, w);
    GRAB_HIP(hipGetLastError());
    if (a.contraction_done) GRAB_HIP(hipEventRecord(a.contraction_done, st));
    ScanFinishArgs f{};
    f.a = a;
    f.list = w.list;
    f.count = w.count;
    f.q_t = q_t;
    f.q_top = q_top;
    f.q_eps = q_eps;
    f.q_norm = q_norm;
    f.q_scale = q_scale;
    f.scal = b.scal;
    f.nq = nq;
    f.k = s.k;
    f.dim = b.dim;
    f.id_bits = w.id_bits;
    if (b.ip) hipLaunchKernelGGL(scan_finish_kernel<kMetricIP>, dim3((nq + 3) / 4), dim3(256), 0, st, f);
    else hipLaunchKernelGGL(scan_finish_kernel<kMetricL2>, dim3((nq + 3) / 4), dim3(256), 0, st, f);
    GRAB_HIP(hipGetLastError());
    return GRAB_OK;
}

}  // namespace grab
