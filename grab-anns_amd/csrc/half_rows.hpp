// Rows rounded to f16 for the matrix pipe, and the queue through which pairs of interest leave it: what knn_half.hip (a row set
// against itself) and scan_half.hip (queries against intervals of a row set) share.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_utils.hpp"
#include "topk_internal.hpp"

namespace grab {
namespace {

using namespace dev;

typedef __attribute__((ext_vector_type(8))) _Float16 v8h;
typedef __attribute__((ext_vector_type(16))) float v16f;
typedef __attribute__((ext_vector_type(4))) uint32_t v4u;  // (arrays of uint4 that a lambda fills end up in scratch memory)

// Layout of packed rows: 32 rows are a block, a block is KS + 1 fragments of 1 KB, a fragment is what one
// v_mfma_f32_32x32x16_f16 takes from the 64 lanes of a wave - 16 bytes each, lane (l32, half) the values k = 16 ks + 8 half
// .. + 7 of row l32.  So every load and every LDS read of a fragment is 1 KB in a row, without padding or conflicts, and
// rows and columns use the same blocks.  The last fragment carries -|row|^2 / 2 as three f16 pieces (33 bits) against
// kNormUnit: a column holds (U, U, U, h0, h1, h2, 0, 0), a row is given (r0, r1, r2, U, U, U, 0, 0) when it is loaded, and
// the accumulator ends up with r + h + row.column.  (Inner product: h = 0, r carries a threshold only.)  Rows of more than 128
// dimensions have a fragment of zeros behind it, which makes their number even.
constexpr float kNormUnit = 16384.0f;
constexpr float kNever = -60000.0f;       // a piece that keeps a padding or non-finite row below every threshold
constexpr float kHalfMin = 6.103515625e-05f;  // smallest normal f16: less becomes zero and counts as remainder
__device__ __forceinline__ float flush_half(float v) { return fabsf(v) < kHalfMin ? 0.0f : v; }
__device__ __forceinline__ uint32_t half_bits(float v) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v); }
__device__ __forceinline__ float half_value(float v) { return (float)(_Float16)v; }
// h / kNormUnit as three f16 pieces
__device__ __forceinline__ void norm_pieces(float h, uint32_t (&p)[3]) {
    float r = h * (1.0f / kNormUnit);
    r = fminf(fmaxf(r, kNever), -kNever);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float v = half_value(flush_half(r));
        p[i] = half_bits(v);
        r -= v;  // exact: v is r's leading bits
    }
}
// 2^e that brings a length of sqrt(max_sq) to [2^12, 2^13)
__device__ __forceinline__ float scale_of(float max_sq) {
    if (!(max_sq > 0.0f)) return 1.0f;
    const int il = ilogbf(max_sq);
    return ldexpf(1.0f, min(max(12 - (il >> 1), -50), 50));
}

// centre[k]: the mean of coordinate k over `count` spaced rows, rounded to a grid of 2^-8 of the coordinate's spread - no
// distance notices which centre is taken, and rows of small integers stay integers on it, which f16 holds exactly.  One
// workgroup per coordinate; zeros beyond dim.
__global__ void __launch_bounds__(256) half_centre_kernel(const float* __restrict__ data, uint64_t n, uint32_t count, uint32_t dim,
                                                          float* __restrict__ centre) {
    __shared__ float s_sum[256], s_min[256], s_max[256];
    const uint32_t k = blockIdx.x, tid = threadIdx.x;
    if (k >= dim) {
        if (tid == 0) centre[k] = 0.0f;
        return;
    }
    float s = 0.0f, lo = __builtin_inff(), hi = -__builtin_inff();
    for (uint32_t i = tid; i < count; i += 256) {
        const float v = data[(size_t)((uint64_t)i * n / count) * dim + k];
        s += v;
        lo = fminf(lo, v);
        hi = fmaxf(hi, v);
    }
    s_sum[tid] = s;
    s_min[tid] = lo;
    s_max[tid] = hi;
    __syncthreads();
    for (uint32_t w = 128; w > 0; w >>= 1) {
        if (tid < w) {
            s_sum[tid] += s_sum[tid + w];
            s_min[tid] = fminf(s_min[tid], s_min[tid + w]);
            s_max[tid] = fmaxf(s_max[tid], s_max[tid + w]);
        }
        __syncthreads();
    }
    if (tid == 0) {
        const float mean = s_sum[0] / (float)count, spread = fmaxf(s_max[0] - mean, mean - s_min[0]);
        float c = mean;
        if (spread > 0.0f && spread < 3.0e38f) {
            const float grid = ldexpf(1.0f, ilogbf(spread) + 1 - 8);
            c = rintf(mean / grid) * grid;
        }
        centre[k] = fabsf(c) < 3.0e38f ? c : 0.0f;  // also where the sample holds infinities or NaN
    }
}

// the largest of the wave's non-negative values into *out; one atomic operation only where it is larger than what stands there
__device__ __forceinline__ void note_largest(float v, uint32_t* out) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
    if ((threadIdx.x & 63) == 0 && __float_as_uint(v) > __atomic_load_n(out, __ATOMIC_RELAXED)) atomicMax(out, __float_as_uint(v));
}

// squared norm of every centred row, and the largest below 3e38, beyond which a row is not packed (scal[0], as bits); scal[kScalLong]:
// whether one is not; 16 lanes a row
__global__ void __launch_bounds__(256) half_norms_kernel(const float* __restrict__ data, uint32_t n, uint32_t dim,
                                                         const float* __restrict__ centre, float* __restrict__ norm, uint32_t* __restrict__ scal) {
    const uint32_t j = threadIdx.x & 15;
    const float4* c4 = reinterpret_cast<const float4*>(centre);
    float most = 0.0f;
    for (uint32_t row = (blockIdx.x * 256 + threadIdx.x) >> 4; row < n; row += gridDim.x * 16) {
        const float4* r4 = reinterpret_cast<const float4*>(data + (size_t)row * dim);
        float s = 0.0f;
        for (uint32_t c = j; c < (dim >> 2); c += 16) {
            const float4 v = r4[c], m = c4[c];
            const float x = v.x - m.x, y = v.y - m.y, z = v.z - m.z, w = v.w - m.w;
            s = __builtin_fmaf(x, x, s);
            s = __builtin_fmaf(y, y, s);
            s = __builtin_fmaf(z, z, s);
            s = __builtin_fmaf(w, w, s);
        }
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) s += __shfl_xor(s, m, 64);
        if (j == 0) norm[row] = s;
        if (j == 0 && s >= 3.0e38f) scal[kScalLong] = 1u;
        if (s < 3.0e38f) most = fmaxf(most, s);
    }
    note_largest(most, scal);
}

// Rows into blocks: place p of the output is row p (kAll), row p * n / count (kSpaced), row perm[p] (kOrdered) or one of 2^count
// rows (kOneOf); places from count (kOneOf: from the last row) on are padding.  hn[p]: squared norm of the rounded, scaled row, -1 for padding and rows that are not finite.
// lift: a power of two on top of the scale.  kAll: eps[row], how far the row moved when it was rounded (unscaled), and the largest of them in scal[1].  16 lanes a row.
enum { kAll = 0, kSpaced = 1, kOrdered = 2, kOneOf = 3 };
// The row that stands for the rows i << shift .. + 2^shift - 1: any of these, not always the first (rows may come in turns).  At
// most 2^31 rows.
__device__ __forceinline__ uint32_t one_of(uint32_t i, uint32_t shift, uint32_t n) { return min((i << shift) + ((i * 0x9E3779B1u) >> (32u - shift)), n - 1u); }
template <int WHICH>
__global__ void __launch_bounds__(256) half_pack_kernel(const float* __restrict__ data, uint64_t n, uint32_t dim, uint32_t ks_count, uint32_t frags,
                                                        float norm_factor, float lift, const float* __restrict__ centre, const float* __restrict__ norm,
                                                        uint32_t* __restrict__ scal, const uint32_t* __restrict__ perm, uint32_t count,
                                                        uint32_t first, uint32_t places, uint4* __restrict__ blocks, float* __restrict__ hn,
                                                        float* __restrict__ eps) {
    const uint32_t p = first + ((blockIdx.x * 256 + threadIdx.x) >> 4), j = threadIdx.x & 15;
    if (p >= places) return;  // whole groups of 16 lanes; places is a multiple of 16
    const float scale = scale_of(__uint_as_float(scal[0])) * lift, unscale = 1.0f / scale;
    const bool live = WHICH == kOneOf ? ((uint64_t)p << count) < n : p < count;
    const uint32_t row = !live ? 0u : WHICH == kSpaced ? (uint32_t)((uint64_t)p * n / count) : WHICH == kOrdered ? perm[p] : WHICH == kOneOf ? one_of(p, count, (uint32_t)n) : p;
    const bool good = live && norm[row] < 3.0e38f;
    const float* x = data + (size_t)row * dim;
    uint4* block = blocks + (size_t)(p >> 5) * frags * 64 + (p & 31);
    float sq = 0.0f, rem = 0.0f;
    for (uint32_t c = j; c < 2 * ks_count; c += 16) {
        uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t k = 8 * c + 4 * h;
            if (good && k < dim) {
                const float4 v = *reinterpret_cast<const float4*>(x + k), m = *reinterpret_cast<const float4*>(centre + k);
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
    if (j < 2) {  // the norm's fragment, and the zeros behind it where there are some
        const uint32_t u = half_bits(kNormUnit);
        uint32_t h[3];
        norm_pieces(good ? norm_factor * sq : kNever * kNormUnit, h);
        block[ks_count * 64 + j * 32] = j == 0 ? make_uint4(u | (u << 16), u | (h[0] << 16), h[1] | (h[2] << 16), 0u) : make_uint4(0u, 0u, 0u, 0u);
        if (frags > ks_count + 1) block[(ks_count + 1) * 64 + j * 32] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (j == 0) hn[p] = good ? sq : -1.0f;
    if (WHICH == kAll) {
        // a little more than the sum's own rounding can hide, and what the subtraction of the centre rounded
        const float e = good ? sqrtf(rem) * unscale * 1.0001f + 1.3e-7f * sqrtf(norm[row]) : 0.0f;
        if (live && j == 0) eps[row] = e;
        note_largest(e, &scal[1]);
        if (live && !good && j == 0) scal[kScalBad] = 1u;
    }
}
// ... a launch has less than 2^32 threads: so many places each
template <int WHICH>
void launch_half_pack(const float* data, uint64_t n, uint32_t dim, uint32_t ks_count, uint32_t frags, float norm_factor, float lift, const float* centre, const float* norm,
                      uint32_t* scal, const uint32_t* perm, uint32_t count, uint32_t places, uint4* blocks, float* hn, float* eps, hipStream_t st) {
    constexpr uint32_t kPlaces = 1u << 27;
    for (uint32_t first = 0; first < places; first += kPlaces)
        hipLaunchKernelGGL(half_pack_kernel<WHICH>, dim3((places - first < kPlaces ? places - first : kPlaces) / 16), dim3(256), 0, st, data, n, dim, ks_count, frags,
                           norm_factor, lift, centre, norm, scal, perm, count, first, places, blocks, hn, eps);
}

// the last fragment of a row as the sweeps want it: lane l32 of the lower half holds row l32's pieces of `h`
__device__ __forceinline__ uint4 row_norm_pieces(float h) {
    const uint32_t u = half_bits(kNormUnit);
    uint32_t p[3];
    norm_pieces(h, p);
    return make_uint4(p[0] | (p[1] << 16), p[2] | (u << 16), u | (u << 16), 0u);
}
__device__ __forceinline__ v8h row_norm_fragment(float h, uint32_t half) {
    return __builtin_bit_cast(v8h, half ? make_uint4(0u, 0u, 0u, 0u) : row_norm_pieces(h));
}
// An entry of a row's list: the column's row number in the low id_bits and above them which part of the way from the largest
// value to the threshold its value lies in, of 2^(32 - id_bits) equal ones - half the bytes of a (distance, row) key, and what
// the finishing kernel wants to know: which few to score.  (Scratch memory that is not asked for matters: memory handed back
// is cleared by the driver in its own time, at some 30 GB/s, and calls that follow each other wait for it once the device's
// memory has gone round.)
__device__ __forceinline__ uint32_t share_of(float g, float t, float top, uint32_t id_bits) {  // t <= g <= top
    const float parts = (float)(1u << (32u - id_bits)), way = top - t;
    const float f = way > 0.0f ? (top - g) / way * parts : 0.0f;
    return (uint32_t)fminf(fmaxf(f, 0.0f), parts - 1.0f) << id_bits;
}

// ---- pairs of interest ----
// An accumulator holds a value less its row's threshold: what is of interest is not negative, and next to nothing is.  A lane
// that has such a value in a block of 32 x 32 copies all its 16 into a queue in LDS; when kQueueAt such entries have gathered
// the wave goes over them, packs the pairs that passed and hands them on, 64 at a time.
constexpr uint32_t kQueueAt = 16;             // entries that set a look at the queue off
constexpr uint32_t kQueueCap = kQueueAt + 64;  // ... and what the block before that look can add
constexpr uint32_t kQueueColumns = 1u << 26;   // a column shares a word with its row block, half and register: it must be less
struct QueueLds {  // a wave's
    uint4 values[kQueueCap * 4];
    uint32_t where[kQueueCap];
    uint2 hits[128];
};
// Sink::put(value, row of the workgroup, column) takes what passed, by as many lanes as there are pairs
template <class Sink>
struct PairQueue {
    Sink sink;
    QueueLds& s;
    const uint32_t lane, first;      // first row of the wave among the workgroup's
    uint32_t queued = 0, found = 0;  // wave-uniform
    __device__ __forceinline__ PairQueue(const Sink& sink_, QueueLds& s_, uint32_t lane_, uint32_t first_) : sink(sink_), s(s_), lane(lane_), first(first_) {}
    __device__ __forceinline__ uint64_t below() const { return (1ull << lane) - 1ull; }

    // `count` pairs (64, or what is left at the end of an item): into the lists of their rows
    __device__ __forceinline__ void append(uint32_t count) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane < count) {
            const uint2 hit = s.hits[lane];
            const uint32_t v = hit.y & 15u, j = hit.y >> 6;
            const uint32_t il = first + ((hit.y >> 5) & 1u) * 32 + (v & 3u) + 8 * (v >> 2) + 4 * ((hit.y >> 4) & 1u);
            sink.put(__uint_as_float(hit.x), il, j);
        }
    }
    // the queued entries, 64 values at a time
    __device__ __forceinline__ void drain() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const uint32_t* vals = reinterpret_cast<const uint32_t*>(s.values);
        for (uint32_t e0 = 0; e0 < queued; e0 += 16) {  // 16 entries, four values a lane
            uint32_t bits[4], where[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {  // (entries past the queue's end hold what an earlier look left)
                bits[u] = vals[(e0 + 4 * u) * 16 + lane];
                where[u] = s.where[e0 + 4 * u + (lane >> 4)];
            }
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const bool pass = (int)bits[u] >= 0 && e0 + 4 * u + (lane >> 4) < queued;
                const uint64_t b = __ballot(pass);
                if (pass) s.hits[found + (uint32_t)__popcll(b & below())] = make_uint2(bits[u], (where[u] << 4) | (lane & 15u));
                found += (uint32_t)__popcll(b);
                if (found >= 64u) {
                    append(64u);
                    __builtin_amdgcn_wave_barrier();
                    const uint2 rest = s.hits[64 + lane];
                    __builtin_amdgcn_wave_barrier();
                    found -= 64u;
                    if (lane < found) s.hits[lane] = rest;
                }
            }
        }
        queued = 0;
        __builtin_amdgcn_wave_barrier();
    }
    // a block of 32 x 32: rows first + 32 rb .. of the tile, this lane's column j < kQueueColumns
    __device__ __forceinline__ void offer(const v16f& acc, uint32_t j, uint32_t rb) {
        int m = -1;
#pragma unroll
        for (uint32_t v = 0; v < 16; v += 2) m = max(max(__float_as_int(acc[v]), __float_as_int(acc[v + 1])), m);
        const uint64_t b = __ballot(m >= 0);
        if (b != 0) {
            if (m >= 0) {
                const uint32_t e = queued + (uint32_t)__popcll(b & below());
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u)
                    s.values[e * 4 + u] = make_uint4(__float_as_uint(acc[4 * u]), __float_as_uint(acc[4 * u + 1]), __float_as_uint(acc[4 * u + 2]),
                                                     __float_as_uint(acc[4 * u + 3]));
                s.where[e] = (j << 2) | (rb << 1) | (lane >> 5);
            }
            queued += (uint32_t)__popcll(b);
            if (queued >= kQueueAt) drain();
        }
    }
    __device__ __forceinline__ void finish() {
        if (queued != 0) drain();
        if (found != 0) append(found);
        found = 0;
    }
};
// 16 bytes a lane from memory to LDS, no registers between: lane l's go to to[l] (`to` the same for the whole wave)
__device__ __forceinline__ void load_to_lds(const v4u* from, v4u* to) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t*)from, (__attribute__((address_space(3))) uint32_t*)to, 16, 0, 0);
}
__device__ __forceinline__ void loads_landed() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0)
}  // namespace
}  // namespace grab
