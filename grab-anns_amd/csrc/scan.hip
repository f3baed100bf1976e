// Exact top-k where a graph is the wrong tool: queries restricted to sets of buckets of a base stored bucket by bucket,
// and queries restricted to intervals of row ids (timestamp windows over rows in timestamp order).  The admitted rows
// are scanned with the contraction kernels of topk_gemm.hip; candidates are re-scored and proven as there.
#include <algorithm>
#include <cstring>
#include <functional>
#include <vector>

#include "common.hpp"
#include "device_sort.hpp"
#include "device_utils.hpp"
#include "topk_gemm.hpp"
#include "topk_internal.hpp"

// ---- exact top-k over sets of buckets, for bases stored bucket by bucket --------------------------------------
namespace grab {
using namespace dev;
namespace {

// row f of dst = row src_row[f] of src (zeros where src_row[f] is 0xFFFFFFFF); 8 lanes per row
__global__ void __launch_bounds__(256) gather_query_rows_kernel(const float* __restrict__ src, const uint32_t* __restrict__ src_row,
                                                                uint32_t count, uint32_t dim, float* __restrict__ dst) {
    const uint32_t g = (blockIdx.x * 256 + threadIdx.x) >> 3;
    const int j = threadIdx.x & 7;
    if (g >= count) return;
    const uint32_t r = src_row[g];
    float4* d4 = reinterpret_cast<float4*>(dst + (size_t)g * dim);
    const float4* s4 = reinterpret_cast<const float4*>(src + (size_t)(r == 0xFFFFFFFFu ? 0 : r) * dim);
    for (uint32_t c = j; c < (dim >> 2); c += 8) d4[c] = r == 0xFFFFFFFFu ? make_float4(0.f, 0.f, 0.f, 0.f) : s4[c];
}

// One wave per query: the k best of the query's partial lists (k sorted results each, -1 where a list ran short),
// by (distance, id).  The lists are taken as many at a time as fit one 1024-key sort beside the best so far.
__global__ void __launch_bounds__(256) merge_partial_lists_kernel(const int64_t* __restrict__ part_ids, const float* __restrict__ part_dist,
                                                                  const uint32_t* __restrict__ list_off, const uint32_t* __restrict__ lists,
                                                                  uint32_t nq, uint32_t k, int64_t* __restrict__ out_ids,
                                                                  float* __restrict__ out_dist) {
    __shared__ uint64_t keys_all[4][1024];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t q = blockIdx.x * 4 + wave;
    if (q >= nq) return;
    uint64_t* keys = keys_all[wave];
    const uint32_t first = list_off[q], last = list_off[q + 1];
    const uint32_t per = (1024u - k) / k;  // lists per round
    for (uint32_t g = lane; g < k; g += 64) keys[g] = kInvalidKey;
    for (uint32_t l0 = first; l0 < last || l0 == first; l0 += per) {
        const uint32_t nl = l0 < last ? min(per, last - l0) : 0u;
        for (uint32_t g = lane; g < 1024u - k; g += 64) {
            uint64_t key = kInvalidKey;
            if (g < nl * k) {
                const size_t at = (size_t)lists[l0 + g / k] * k + g % k;
                const int64_t id = part_ids[at];
                if (id >= 0) key = make_sel_key(part_dist[at], (uint32_t)id);
            }
            keys[k + g] = key;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint64_t r[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) r[i] = keys[lane * 16 + i];
        wave_bitonic_sort<16>(r);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if ((uint32_t)(lane * 16 + i) < k) keys[lane * 16 + i] = r[i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (nl == 0) break;
    }
    for (uint32_t g = lane; g < k; g += 64) {
        const uint64_t key = keys[g];
        const bool valid = key != kInvalidKey;
        out_ids[(size_t)q * k + g] = valid ? (int64_t)(key & 0xFFFFFFFFull) : -1;
        out_dist[(size_t)q * k + g] = valid ? ord_float((uint32_t)(key >> 32)) : kDistMax;
    }
}

// One wave per query: the query's candidate lists - `splits` lists of kk GEMM-form keys for each of its tile-grid rows,
// each the kk smallest of its slice of columns - become one ascending list of the kk smallest.  outside[q] = the
// smallest last key of a full list: every column that is in no list lies at or beyond it (what the merge itself
// drops shows in the merged list's own last key).
__global__ void __launch_bounds__(256) premerge_lists_kernel(const uint64_t* __restrict__ cand, uint32_t splits, uint32_t kk,
                                                             const uint32_t* __restrict__ list_off, const uint32_t* __restrict__ lists,
                                                             uint32_t nq, uint64_t* __restrict__ merged, float* __restrict__ outside) {
    __shared__ uint64_t keys_all[4][1024];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t q = blockIdx.x * 4 + wave;
    if (q >= nq) return;
    uint64_t* keys = keys_all[wave];
    const uint32_t first = list_off[q], total = (list_off[q + 1] - first) * splits;
    const uint32_t per = (1024u - kk) / kk;  // lists per round (kk <= 512)
    auto list_base = [&](uint32_t li) { return cand + ((size_t)lists[first + li / splits] * splits + li % splits) * kk; };
    for (uint32_t g = lane; g < kk; g += 64) keys[g] = kInvalidKey;
    float out = __builtin_inff();
    for (uint32_t l0 = 0; l0 < total; l0 += per) {
        const uint32_t nl = min(per, total - l0);
        for (uint32_t g = lane; g < 1024u - kk; g += 64) keys[kk + g] = g < nl * kk ? list_base(l0 + g / kk)[g % kk] : kInvalidKey;
        if ((uint32_t)lane < nl) {
            const uint64_t last = list_base(l0 + lane)[kk - 1];
            if (last != kInvalidKey) out = fminf(out, ord_float((uint32_t)(last >> 32)));
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint64_t r[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) r[i] = keys[lane * 16 + i];
        wave_bitonic_sort<16>(r);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if ((uint32_t)(lane * 16 + i) < kk) keys[lane * 16 + i] = r[i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) out = fminf(out, __shfl_xor(out, m, 64));
    for (uint32_t g = lane; g < kk; g += 64) merged[(size_t)q * kk + g] = keys[g];
    if (lane == 0) outside[q] = out;
}

// results of a subset of the queries back to their places
__global__ void __launch_bounds__(256) scatter_results_kernel(const int64_t* __restrict__ ids, const float* __restrict__ dist,
                                                              const uint32_t* __restrict__ rows, uint32_t count, uint32_t k,
                                                              int64_t* __restrict__ out_ids, float* __restrict__ out_dist) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= count * k) return;
    const size_t at = (size_t)rows[i / k] * k + i % k;
    out_ids[at] = ids[i];
    out_dist[at] = dist[i];
}

// The key of lane ^ MASK, without a trip to LDS up to 15.
template <int MASK>
__device__ __forceinline__ uint64_t lane_xor_u64(uint64_t v) {
    const int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
    auto dpp = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        return ((uint64_t)(uint32_t)__builtin_amdgcn_update_dpp(hi, hi, C, 0xF, 0xF, false) << 32) |
               (uint32_t)__builtin_amdgcn_update_dpp(lo, lo, C, 0xF, 0xF, false);
    };
    if constexpr (MASK == 1) return dpp(std::integral_constant<int, 0xB1>{});        // quad_perm 1 0 3 2
    else if constexpr (MASK == 2) return dpp(std::integral_constant<int, 0x4E>{});   // quad_perm 2 3 0 1
    else if constexpr (MASK == 3) return dpp(std::integral_constant<int, 0x1B>{});   // quad_perm 3 2 1 0
    else if constexpr (MASK == 4) return lane_xor_u64<3>(lane_xor_u64<7>(v));
    else if constexpr (MASK == 7) return dpp(std::integral_constant<int, 0x141>{});  // row_half_mirror
    else if constexpr (MASK == 8) return dpp(std::integral_constant<int, 0x128>{});  // row_ror 8
    else if constexpr (MASK == 15) return dpp(std::integral_constant<int, 0x140>{}); // row_mirror
    else return shfl_xor_u64(v, MASK);
}
// lanes that differ in MASK: the one without BIT (the highest of MASK) keeps the smaller key
template <int MASK, int BIT>
__device__ __forceinline__ void order_pair(uint64_t& k, int lane) {
    const uint64_t o = lane_xor_u64<MASK>(k);
    k = (k < o) == ((lane & BIT) == 0) ? k : o;
}
// a run of S lanes that first rises, then falls (or the other way) becomes ascending; S = 2 * BIT
template <int BIT>
__device__ __forceinline__ void bitonic_halves(uint64_t& k, int lane) {
    order_pair<BIT, BIT>(k, lane);
    if constexpr (BIT > 1) bitonic_halves<BIT / 2>(k, lane);
}
template <int SIZE>
__device__ __forceinline__ void sort_merge_runs(uint64_t& k, int lane) {  // ascending runs of SIZE / 2 lanes to runs of SIZE
    order_pair<SIZE - 1, SIZE / 2>(k, lane);
    if constexpr (SIZE > 2) bitonic_halves<SIZE / 4>(k, lane);
}
__device__ __forceinline__ void sort_lanes(uint64_t& k, int lane) {  // one key a lane, ascending
    sort_merge_runs<2>(k, lane);
    sort_merge_runs<4>(k, lane);
    sort_merge_runs<8>(k, lane);
    sort_merge_runs<16>(k, lane);
    sort_merge_runs<32>(k, lane);
    sort_merge_runs<64>(k, lane);
}

// The same walk for the exact scans: one wave per tile-grid row of the distances that the contraction left, a row tile as
// wide as its sweep (sched holds where it starts, in the matrix and among the columns).  The kk (<= 64) smallest
// (distance, column) keys of the row's columns [lo, hi) go to keys[query][kk] in ascending order, or to keys[row][kk]
// without row_query; rows that admit no column are padding.
// Bound by instruction issue.  What passes the threshold - the list's kk-th key - gathers in LDS and is sorted and merged
// into the list 64 keys at a time: a threshold that lags lets a few more keys pass (some 64 for every doubling of the
// columns seen), but a key costs four instructions of a sort instead of the two dozen of an insertion of its own.  10,000
// intervals of 10,000 columns (0.4 GB): 190 -> 127 us; 200k x 768 in 64 buckets, 16,500 lists: 160 -> 81 us.
__global__ void __launch_bounds__(256) stream_select_keys_kernel(const float* __restrict__ dense, const uint32_t* __restrict__ row_query, const uint32_t* __restrict__ row_lo,
                                                                 const uint32_t* __restrict__ row_hi, const uint32_t* __restrict__ sched,
                                                                 uint32_t nrows, uint32_t kk, uint64_t* __restrict__ out_keys) {
    const int lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= nrows) return;
    const uint32_t c_lo = row_lo[row], c_hi = row_hi[row];
    if (c_lo >= c_hi) return;
    const uint32_t base = sched[kSchedLo + row / TM] * TN;  // <= c_lo: the row tile's sweep starts at or before every interval of its rows
    const uint32_t tile = row / TM;
    const uint32_t pitch = (sched[kSchedHi + tile] - sched[kSchedLo + tile]) * TN;
    const float* drow = dense + (size_t)sched[kSchedBase + tile] * (TM * TN) + (size_t)(row % TM) * pitch;
    __shared__ uint64_t waiting_all[4][128];
    uint64_t* waiting = waiting_all[threadIdx.x >> 6];
    uint32_t nwait = 0;  // wave-uniform, below 64 between offers
    uint64_t mykey = kInvalidKey;
    float thr_d = __builtin_inff();
    auto merge_waiting = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint64_t x = (uint32_t)lane < nwait ? waiting[lane] : kInvalidKey;
        const uint64_t rest = waiting[64 + lane];
        sort_lanes(x, lane);
        const uint64_t o = lane_xor_u64<63>(x);
        mykey = mykey < o ? mykey : o;  // the 64 smallest of both
        bitonic_halves<32>(mykey, lane);
        const uint64_t thr = readlane_u64(mykey, (int)kk - 1);
        const float d = ord_float((uint32_t)(thr >> 32));
        thr_d = thr == kInvalidKey || d != d ? __builtin_inff() : d;
        nwait = nwait > 64u ? nwait - 64u : 0u;
        __builtin_amdgcn_wave_barrier();
        if ((uint32_t)lane < nwait) waiting[lane] = rest;
    };
    auto offer = [&](bool pass, float d, uint32_t c) {
        const uint64_t b = __ballot(pass);
        if (b == 0) return;
        if (pass) waiting[nwait + (uint32_t)__popcll(b & ((1ull << lane) - 1ull))] = make_sel_key(d, c);
        nwait += (uint32_t)__popcll(b);
        if (nwait >= 64u) merge_waiting();
    };
    // of an interval of 512 columns and more the first 512 are all candidates, those without an order (NaN) among them; a
    // bucket's row takes none of these, like the selection inside the contraction that longer lists go through
    const uint32_t c_from = row_query != nullptr && c_hi - c_lo >= 512u ? c_lo + 512u : c_lo;
    // 512 columns per step, two runs of four consecutive columns per lane, the next step's loads issued before this
    // step's values are looked at; steps are aligned to the row's first stored column
    constexpr uint32_t STEP = 512;
    const uint32_t c_begin = base + ((c_lo - base) & ~(STEP - 1));
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load4 = [&](uint32_t c) { return c < c_hi ? *reinterpret_cast<const float4*>(drow + (c - base)) : zero; };
    float4 cur0 = load4(c_begin + 4 * lane), cur1 = load4(c_begin + 256 + 4 * lane);
    for (uint32_t c0 = c_begin; c0 < c_hi; c0 += STEP) {
        float4 nxt0 = zero, nxt1 = zero;
        if (c0 + STEP < c_hi) {
            nxt0 = load4(c0 + STEP + 4 * lane);
            nxt1 = load4(c0 + STEP + 256 + 4 * lane);
        }
        const float dv[8] = {cur0.x, cur0.y, cur0.z, cur0.w, cur1.x, cur1.y, cur1.z, cur1.w};
        const bool interior = c0 >= c_from && c0 + STEP <= c_hi;  // wave-uniform
        if (interior) {
            bool any = false;
#pragma unroll
            for (int e = 0; e < 8; ++e) any = any || dv[e] <= thr_d;
            if (__ballot(any) != 0) {
#pragma unroll
                for (int e = 0; e < 8; ++e) offer(dv[e] <= thr_d, dv[e], c0 + (e >> 2) * 256 + 4 * lane + (e & 3));
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t c = c0 + (e >> 2) * 256 + 4 * lane + (e & 3);
                offer(c >= c_lo && c < c_hi && (dv[e] <= thr_d || (c < c_from && dv[e] != dv[e])), dv[e], c);
            }
        }
        cur0 = nxt0;
        cur1 = nxt1;
    }
    if (nwait != 0) merge_waiting();
    if ((uint32_t)lane < kk) out_keys[(size_t)(row_query ? row_query[row] : row) * kk + lane] = mykey;
}

constexpr uint32_t kScanPiece = 128 * TN;  // columns of one piece of a bucket: a work item sweeps at most this many

// What both ways of the bucket scan work on: every (query, bucket of the query) pair is a tile-grid row with the
// bucket's rows as its admissible columns; a long bucket is cut into pieces, a row per piece.  The rows of a piece
// follow each other, padded to whole row tiles (with rows that admit no column): a tile visits its piece's columns only.
struct ScanRows {
    struct Piece {
        uint32_t lo, hi;
    };
    std::vector<Piece> pieces;
    std::vector<uint32_t> piece_row0;                  // first row of each piece
    std::vector<uint32_t> row_query, row_lo, row_hi;   // per tile-grid row
    std::vector<uint32_t> list_off, lists;             // per query: its tile-grid rows
    uint32_t rows = 0;
    double tiles = 0.0;                                // (row tile, column tile) pairs that the sweep visits
    std::vector<uint32_t> tile_lo, tile_hi;            // per row tile the column tiles [lo, hi) that its rows admit
    bool one_row_per_query = false;                    // id intervals: row tiles in the order of the intervals' starts
    uint64_t columns = 0, widest = 0;                  // ... and what the intervals admit in all, and the widest of them
};

void scan_rows(const uint64_t* h_bucket_offsets, uint32_t num_buckets, const uint64_t* h_masks, size_t num_queries, ScanRows* out) {
    ScanRows& r = *out;
    std::vector<uint32_t> first_piece(num_buckets + 1, 0);
    for (uint32_t b = 0; b < num_buckets; ++b) {
        first_piece[b] = (uint32_t)r.pieces.size();
        for (uint64_t s0 = h_bucket_offsets[b]; s0 < h_bucket_offsets[b + 1]; s0 += kScanPiece)
            r.pieces.push_back({(uint32_t)s0, (uint32_t)std::min<uint64_t>(s0 + kScanPiece, h_bucket_offsets[b + 1])});
    }
    first_piece[num_buckets] = (uint32_t)r.pieces.size();
    // a query's set is walked along its set bits, not bucket by bucket (a branch that is rarely foretold, twice per query and
    // bucket): the device waits for these tables.  4999 queries of 1-4 of 64 buckets: call 1.01 -> 0.67 ms
    const uint64_t known = num_buckets == 64 ? ~0ull : (1ull << num_buckets) - 1ull;
    std::vector<uint32_t> piece_count(r.pieces.size() + 1, 0);
    r.list_off.assign(num_queries + 1, 0);
    for (size_t q = 0; q < num_queries; ++q) {
        uint32_t n = 0;
        for (uint64_t m = h_masks[q] & known; m != 0; m &= m - 1) {
            const uint32_t b = (uint32_t)__builtin_ctzll(m);
            for (uint32_t pc = first_piece[b]; pc < first_piece[b + 1]; ++pc) piece_count[pc + 1]++;
            n += first_piece[b + 1] - first_piece[b];
        }
        r.list_off[q + 1] = r.list_off[q] + n;
    }
    r.piece_row0.assign(r.pieces.size() + 1, 0);
    for (size_t pc = 0; pc < r.pieces.size(); ++pc) r.piece_row0[pc + 1] = r.piece_row0[pc] + (piece_count[pc + 1] + TM - 1) / TM * TM;
    r.rows = r.piece_row0[r.pieces.size()];
    r.row_query.assign(r.rows, 0u);  // padding rows stand for query 0 and admit no column
    r.row_lo.assign(r.rows, 0);
    r.row_hi.assign(r.rows, 0);
    r.lists.resize(r.list_off[num_queries]);
    std::vector<uint32_t> fill(r.piece_row0.begin(), r.piece_row0.end() - 1), at(r.list_off.begin(), r.list_off.end() - 1);
    for (size_t q = 0; q < num_queries; ++q)
        for (uint64_t m = h_masks[q] & known; m != 0; m &= m - 1) {
            const uint32_t b = (uint32_t)__builtin_ctzll(m);
            for (uint32_t pc = first_piece[b]; pc < first_piece[b + 1]; ++pc) {
                const uint32_t row = fill[pc]++;
                r.row_query[row] = (uint32_t)q;
                r.row_lo[row] = r.pieces[pc].lo;
                r.row_hi[row] = r.pieces[pc].hi;
                r.lists[at[q]++] = row;
            }
        }
    for (size_t pc = 0; pc < r.pieces.size(); ++pc) {
        const uint32_t lo = r.pieces[pc].lo / TN, hi = (r.pieces[pc].hi + TN - 1) / TN;
        for (uint32_t row = r.piece_row0[pc]; row < r.piece_row0[pc + 1]; row += TM) {
            r.tiles += hi - lo;
            r.tile_lo.push_back(lo);
            r.tile_hi.push_back(hi);
        }
    }
}

// Id intervals instead of buckets: a query is one tile-grid row whose admissible columns are its interval.  The queries
// go into the row tiles in the order of their intervals' starts, so that a tile - which sweeps the union of its rows'
// intervals - visits few columns that none of its rows admits.  `which`: the queries meant (numbered 0.. in the result), or
// null for all.  A query with an empty interval gets no row.
void window_rows(const uint64_t* h_lo, const uint64_t* h_hi, const uint32_t* which, size_t count, size_t num_dataset, ScanRows* out) {
    ScanRows& r = *out;
    struct Item {
        uint32_t lo, hi, q;
    };
    std::vector<Item> items;
    items.reserve(count);
    for (size_t i = 0; i < count; ++i) {
        const size_t src = which ? which[i] : i;
        const uint64_t lo = std::min<uint64_t>(h_lo[src], num_dataset), hi = std::min<uint64_t>(h_hi[src], num_dataset);
        if (lo < hi) {
            items.push_back({(uint32_t)lo, (uint32_t)hi, (uint32_t)i});
            r.columns += hi - lo;
            r.widest = std::max(r.widest, hi - lo);
        }
    }
    {   // by (start, end, query): a counting pass over 4096 stretches of the starts, then the few items of a stretch
        constexpr uint32_t kBins = 4096;
        std::vector<uint32_t> first(kBins + 1, 0);
        auto bin = [&](const Item& it) { return (uint32_t)(((uint64_t)it.lo * kBins) / (num_dataset + 1)); };
        for (const Item& it : items) first[bin(it) + 1]++;
        for (uint32_t b = 0; b < kBins; ++b) first[b + 1] += first[b];
        std::vector<Item> placed(items.size());
        std::vector<uint32_t> at(first.begin(), first.end() - 1);
        for (const Item& it : items) placed[at[bin(it)]++] = it;
        for (uint32_t b = 0; b < kBins; ++b)
            if (first[b + 1] - first[b] > 1)
                std::sort(placed.begin() + first[b], placed.begin() + first[b + 1],
                          [](const Item& a, const Item& b) { return a.lo != b.lo ? a.lo < b.lo : (a.hi != b.hi ? a.hi < b.hi : a.q < b.q); });
        items.swap(placed);
    }
    r.rows = (uint32_t)((items.size() + TM - 1) / TM * TM);
    r.row_query.assign(r.rows, 0u);  // padding rows stand for query 0 and admit no column
    r.row_lo.assign(r.rows, 0);
    r.row_hi.assign(r.rows, 0);
    r.list_off.assign(count + 1, 0);
    for (const Item& it : items) r.list_off[it.q + 1] = 1;
    for (size_t q = 0; q < count; ++q) r.list_off[q + 1] += r.list_off[q];
    r.lists.assign(items.size(), 0u);
    for (size_t row = 0; row < items.size(); ++row) {
        r.row_query[row] = items[row].q;
        r.row_lo[row] = items[row].lo;
        r.row_hi[row] = items[row].hi;
        r.lists[r.list_off[items[row].q]] = (uint32_t)row;
    }
    for (size_t row0 = 0; row0 < items.size(); row0 += TM) {
        uint32_t lo = 0xFFFFFFFFu, hi = 0;
        for (size_t row = row0; row < std::min(items.size(), row0 + TM); ++row) {
            lo = std::min(lo, items[row].lo);
            hi = std::max(hi, items[row].hi);
        }
        r.tiles += (double)((hi + TN - 1) / TN - lo / TN);
        r.tile_lo.push_back(lo / TN);
        r.tile_hi.push_back((hi + TN - 1) / TN);
    }
    r.one_row_per_query = true;
}

// The plain way: every tile-grid row is a problem of its own for exact_topk (the query's row gathered once per
// tile-grid row, candidates re-scored and checked per row), and a query's partial results are merged at the end.
// Takes what the quick way below cannot prove.
int bucket_scan_by_rows(const float* d_dataset, size_t num_dataset, uint32_t dim, const ScanRows& r, const float* d_queries,
                        size_t num_queries, uint32_t k, int metric, int64_t* d_out_indices, float* d_out_dists, hipStream_t st) {
    DeviceScratch d_rq, d_lo, d_hi, d_rows, d_pid, d_pdist, d_loff, d_lists;
    const uint32_t rows = r.rows;
    GRAB_HIP(d_rq.alloc((size_t)rows * 4));
    GRAB_HIP(d_lo.alloc((size_t)rows * 4));
    GRAB_HIP(d_hi.alloc((size_t)rows * 4));
    GRAB_HIP(d_rows.alloc((size_t)rows * dim * 4));
    GRAB_HIP(d_pid.alloc((size_t)rows * k * 8));
    GRAB_HIP(d_pdist.alloc((size_t)rows * k * 4));
    GRAB_HIP(d_loff.alloc(r.list_off.size() * 4));
    GRAB_HIP(d_lists.alloc(std::max<size_t>(r.lists.size(), 1) * 4));
    GRAB_HIP(hipMemcpyAsync(d_rq.ptr, r.row_query.data(), (size_t)rows * 4, hipMemcpyHostToDevice, st));
    GRAB_HIP(hipMemcpyAsync(d_lo.ptr, r.row_lo.data(), (size_t)rows * 4, hipMemcpyHostToDevice, st));
    GRAB_HIP(hipMemcpyAsync(d_hi.ptr, r.row_hi.data(), (size_t)rows * 4, hipMemcpyHostToDevice, st));
    GRAB_HIP(hipMemcpyAsync(d_loff.ptr, r.list_off.data(), r.list_off.size() * 4, hipMemcpyHostToDevice, st));
    if (!r.lists.empty()) GRAB_HIP(hipMemcpyAsync(d_lists.ptr, r.lists.data(), r.lists.size() * 4, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(gather_query_rows_kernel, dim3((uint32_t)(((size_t)rows * 8 + 255) / 256)), dim3(256), 0, st, d_queries,
                       d_rq.as<uint32_t>(), rows, dim, d_rows.as<float>());
    GRAB_HIP(hipGetLastError());
    TopkProblem p{};
    p.A = d_rows.as<float>();
    p.B = d_dataset;
    p.M = rows;
    p.N = num_dataset;
    p.dim = dim;
    p.k = k;
    p.metric = metric;
    p.filter_kind = kFilterColRange;
    p.row_lo = d_lo.as<uint32_t>();
    p.row_hi = d_hi.as<uint32_t>();
    p.out_i64 = d_pid.as<int64_t>();
    p.out_dist = d_pdist.as<float>();
    GRAB_TRY(exact_topk(p, st, nullptr));
    hipLaunchKernelGGL(merge_partial_lists_kernel, dim3((uint32_t)((num_queries + 3) / 4)), dim3(256), 0, st, d_pid.as<int64_t>(),
                       d_pdist.as<float>(), d_loff.as<uint32_t>(), d_lists.as<uint32_t>(), (uint32_t)num_queries, k, d_out_indices,
                       d_out_dists);
    GRAB_HIP(hipGetLastError());
    GRAB_HIP(hipStreamSynchronize(st));  // the partial lists are freed on return
    return GRAB_OK;
}


// the base rows as bf16 halves, centred on a mean of spaced rows for squared L2 (mean_out receives it), and their norms
int split_base_rows(const float* d_dataset, size_t num_dataset, uint32_t dim, int metric, DeviceScratch* mean_out, uint16_t* d_split,
                    float* d_norm, hipStream_t st) {
    const float* mu = nullptr;
    if (metric == kMetricL2) {
        GRAB_HIP(mean_out->alloc((size_t)dim * 4));
        launch_spaced_mean(d_dataset, num_dataset, (uint32_t)std::min<size_t>(num_dataset, 8192), dim, mean_out->as<float>(), st);
        mu = mean_out->as<float>();
    }
    launch_split_rows_chunked(d_dataset, num_dataset, dim, mu, d_split, d_norm, st);
    GRAB_HIP(hipGetLastError());
    return GRAB_OK;
}

// What a scan needs of the base rows and can keep between calls: the rows as bf16 halves (centred on `mean` for squared
// L2) or as they are, their squared norms (of the centred rows where centred) and the largest of these.
struct ScanBase {
    bool split = false;
    const uint16_t* rows_split = nullptr;
    const float* norm = nullptr;
    const float* mean = nullptr;      // null: not centred
    const float* max_norm = nullptr;  // one float
    void** staging = nullptr;         // page-locked host memory for a call's tables, grown as needed (null: none kept)
    size_t* staging_bytes = nullptr;
    const HalfBase* half = nullptr;   // the rows rounded to f16, where these are what a call uses first
    std::function<int(hipStream_t, bool* no_room)> make_split;  // ... and rows_split is made when a call needs it after all
};

// A call's tables, put together on the host and brought to the device in one upload
struct ScanUpload {
    std::vector<uint32_t> tab;
    size_t put(const uint32_t* src, size_t count) {  // every table starts on a 64-byte boundary
        tab.resize((tab.size() + 15) / 16 * 16);
        const size_t at = tab.size();
        tab.insert(tab.end(), src, src + count);
        return at;
    }
    int upload(const ScanBase* base, DeviceScratch* d_tab, hipStream_t st) {
        GRAB_HIP(d_tab->alloc(tab.size() * 4 + 64));
        // a prepared base keeps page-locked memory for the tables: the upload is queued and the host goes on (from
        // pageable memory the call waits for the copy)
        const void* src = tab.data();
        if (base && base->staging) {
            if (*base->staging_bytes < tab.size() * 4) {
                if (*base->staging) (void)hipHostFree(*base->staging);
                *base->staging = nullptr;
                *base->staging_bytes = 0;
                const size_t want = tab.size() * 4 + tab.size() + 4096;
                if (hipHostMalloc(base->staging, want, hipHostMallocDefault) == hipSuccess) *base->staging_bytes = want;
                else (void)hipGetLastError();
            }
            if (*base->staging) {
                std::memcpy(*base->staging, tab.data(), tab.size() * 4);
                src = *base->staging;
            }
        }
        GRAB_HIP(hipMemcpyAsync(d_tab->ptr, src, tab.size() * 4, hipMemcpyHostToDevice, st));
        return GRAB_OK;
    }
};

// what a call starts from: no row unproven yet, no largest norm yet, the work counters of its launches at zero, every
// candidate list empty (`keys` may be null)
__global__ void __launch_bounds__(256) scan_init_kernel(uint32_t* __restrict__ doubt, uint32_t nq, uint32_t counters, uint64_t* __restrict__ keys, size_t count) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i == 0) {
        doubt[0] = 0;
        doubt[nq + 1] = 0;
        doubt[nq + 2] = 0;
    }
    if (i < counters) doubt[nq + 3 + i] = 0;
    for (size_t g = i; g < count; g += (size_t)gridDim.x * 256) keys[g] = kInvalidKey;
}

// The work list of the dense-store contraction for row tiles whose column tiles [lo, hi) are known on the host: items of
// `per` column tiles, priced like bucket_order_kernel prices them (rounds of `grid` concurrent items, each costing its
// tiles plus a start-up of about a third of a tile).
void dense_sched(const uint32_t* tile_lo, const uint32_t* tile_hi, uint32_t row_tiles, uint32_t grid, uint32_t* sched) {
    uint32_t total = 0;
    for (uint32_t t = 0; t < row_tiles; ++t) total += tile_hi[t] - tile_lo[t];
    const uint32_t base = std::max(1u, total / (grid * 8u));
    uint32_t per = base, best = 0xFFFFFFFFu;
    for (uint32_t w = 0; w < 16; ++w) {
        const uint32_t cand = base + w;
        uint32_t n = 0;
        for (uint32_t t = 0; t < row_tiles; ++t) n += (tile_hi[t] - tile_lo[t] + cand - 1) / cand;
        const uint32_t cost = ((n + grid - 1) / grid) * (3 * cand + 1);
        if (cost < best) {
            best = cost;
            per = cand;
        }
    }
    uint32_t acc = 0, tiles = 0;
    for (uint32_t t = 0; t < row_tiles; ++t) {
        sched[kSchedOff + t] = acc;
        sched[kSchedLo + t] = tile_lo[t];
        sched[kSchedHi + t] = tile_hi[t];
        sched[kSchedBase + t] = tiles;
        tiles += tile_hi[t] - tile_lo[t];
        acc += (tile_hi[t] - tile_lo[t] + per - 1) / per;
    }
    sched[kSchedOff + row_tiles] = acc;
    sched[kSchedPer] = per;
    sched[kSchedItems] = acc;
}

// What the quick way needs beyond the rows: the rows of a subset of the queries (ascending query numbers), for the plain way.
using SubRows = std::function<void(const std::vector<uint32_t>& which, ScanRows* out)>;

enum RowsAs { kOnF16, kAsHalves, kAsTheyAre };  // on f16 rows wherever these serve; as two bf16 halves where the base has or makes them, or at once
int scan_topk(const float* d_dataset, size_t num_dataset, uint32_t dim, const ScanRows& rw, const SubRows& sub_rows, const float* d_queries, size_t num_queries,
              uint32_t k, int metric, int64_t* d_out_indices, float* d_out_dists, float* kernel_ms, hipStream_t st, const ScanBase* base, RowsAs rows_as);

// Queries that a pass could not prove, doubt[1 .. n_doubt]: all those of a pass on f16 rows once more (rows_as other than kOnF16; base: the
// call's), the plain way after any other pass.
int unproven_queries(const float* d_dataset, size_t num_dataset, uint32_t dim, const SubRows& sub_rows, const float* d_queries, uint32_t k, int metric,
                     const uint32_t* doubt, uint32_t n_doubt, int64_t* d_out_indices, float* d_out_dists, hipStream_t st, RowsAs rows_as = kOnF16,
                     const ScanBase* base = nullptr) {
    std::vector<uint32_t> which(n_doubt);
    GRAB_HIP(hipMemcpy(which.data(), doubt + 1, (size_t)n_doubt * 4, hipMemcpyDeviceToHost));
    std::sort(which.begin(), which.end());
    ScanRows sub;
    sub_rows(which, &sub);
    DeviceScratch d_which, sub_q, sub_ids, sub_dist;
    GRAB_HIP(d_which.alloc((size_t)n_doubt * 4));
    GRAB_HIP(sub_q.alloc((size_t)n_doubt * dim * 4));
    GRAB_HIP(sub_ids.alloc((size_t)n_doubt * k * 8));
    GRAB_HIP(sub_dist.alloc((size_t)n_doubt * k * 4));
    GRAB_HIP(hipMemcpyAsync(d_which.ptr, which.data(), (size_t)n_doubt * 4, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(gather_query_rows_kernel, dim3((uint32_t)(((size_t)n_doubt * 8 + 255) / 256)), dim3(256), 0, st, d_queries,
                       d_which.as<uint32_t>(), n_doubt, dim, sub_q.as<float>());
    GRAB_HIP(hipGetLastError());
    const KnnStats main_pass = knn_stats();
    const bool again = rows_as != kOnF16;
    if (again) {
        const SubRows of_these = [&](const std::vector<uint32_t>& some, ScanRows* out) {
            std::vector<uint32_t> of_call(some);
            for (uint32_t& q : of_call) q = which[q];
            sub_rows(of_call, out);
        };
        GRAB_TRY(scan_topk(d_dataset, num_dataset, dim, sub, of_these, sub_q.as<float>(), n_doubt, k, metric, sub_ids.as<int64_t>(), sub_dist.as<float>(), nullptr,
                           st, base, rows_as));
    } else {
        GRAB_TRY(bucket_scan_by_rows(d_dataset, num_dataset, dim, sub, sub_q.as<float>(), n_doubt, k, metric, sub_ids.as<int64_t>(),
                                     sub_dist.as<float>(), st));
    }
    const uint64_t exact = again ? knn_stats().exact_rows : n_doubt;
    knn_stats() = main_pass;  // the figures of the main pass
    knn_stats().exact_rows = main_pass.exact_rows + exact;
    if (again) knn_stats().redone_rows += n_doubt;
    hipLaunchKernelGGL(scatter_results_kernel, dim3((n_doubt * k + 255) / 256), dim3(256), 0, st, sub_ids.as<int64_t>(), sub_dist.as<float>(),
                       d_which.as<uint32_t>(), n_doubt, k, d_out_indices, d_out_dists);
    GRAB_HIP(hipGetLastError());
    GRAB_HIP(hipStreamSynchronize(st));
    return GRAB_OK;
}

// the results of queries of which none admits a row
int no_row_admitted(size_t num_queries, uint32_t k, int64_t* d_out_indices, float* d_out_dists, hipStream_t st) {
    std::vector<int64_t> ids(num_queries * (size_t)k, -1);
    std::vector<float> dist(num_queries * (size_t)k, kDistMax);
    GRAB_HIP(hipMemcpyAsync(d_out_indices, ids.data(), ids.size() * 8, hipMemcpyHostToDevice, st));
    GRAB_HIP(hipMemcpyAsync(d_out_dists, dist.data(), dist.size() * 4, hipMemcpyHostToDevice, st));
    GRAB_HIP(hipStreamSynchronize(st));
    return GRAB_OK;
}

// One pass of the f16 way (scan_half.hip) over queries [first, first + nq) of the call, whose rows are `rw`; its kernels' time is added
// to *kernel_ms.  *applied = false: a query or a row that this way does not take, or no room.
constexpr size_t kHalfPassBytes = (size_t)4 << 30;  // device memory of a pass: what the other way's passes take
constexpr uint32_t kHalfPassQueries = 128;          // ... which fewer queries than these are not split for
int scan_half_pass(const HalfBase& b, const float* d_dataset, size_t num_dataset, const ScanRows& rw, const SubRows& sub_rows, const float* d_queries, uint32_t first,
                   uint32_t nq, uint32_t k, int metric, int64_t* d_out_indices, float* d_out_dists, float* kernel_ms, hipStream_t st, const ScanBase* base,
                   uint32_t num_cu, bool* applied) {
    const uint32_t rows = rw.rows, dim = b.dim;
    *applied = rows == 0;  // (a part of a call may be without any)
    if (rows == 0) return no_row_admitted(nq, k, d_out_indices + (size_t)first * k, d_out_dists + (size_t)first * k, st);
    HalfScan s;
    s.rows = rows;
    s.nq = nq;
    s.k = k;
    s.tile_lo = rw.tile_lo.data();
    s.tile_hi = rw.tile_hi.data();
    if (!half_scan_plan(b, num_cu, rw.row_lo.data(), rw.row_hi.data(), kHalfPassBytes, &s)) {
        if (nq <= kHalfPassQueries) return GRAB_OK;
        for (uint32_t part = 0; part < 2; ++part) {
            const uint32_t from = part == 0 ? first : first + nq / 2, count = part == 0 ? nq / 2 : nq - nq / 2;
            std::vector<uint32_t> which(count);
            for (uint32_t i = 0; i < count; ++i) which[i] = from + i;
            ScanRows half;
            sub_rows(which, &half);
            GRAB_TRY(scan_half_pass(b, d_dataset, num_dataset, half, sub_rows, d_queries, from, count, k, metric, d_out_indices, d_out_dists, kernel_ms, st, base, num_cu,
                                    applied));
            if (!*applied) return GRAB_OK;
        }
        return GRAB_OK;
    }
    struct Rewind {  // a pass is through with its scratch when it returns: the next one gets the same
        ScratchArena* const arena = scratch_arena();
        const size_t used = arena ? arena->used : 0, wanted = arena ? arena->wanted : 0;
        ~Rewind() {
            if (!arena) return;
            arena->peak = std::max(arena->peak, arena->wanted);
            arena->used = used;
            arena->wanted = wanted;
        }
    } rewind;
    DeviceScratch d_tab, ws;
    ScanUpload up;
    up.tab.reserve((size_t)rows * 3 + rw.list_off.size() + rw.lists.size() + s.words.size() + 96);
    const size_t at_rq = up.put(rw.row_query.data(), rows), at_lo = up.put(rw.row_lo.data(), rows), at_hi = up.put(rw.row_hi.data(), rows);
    const size_t at_loff = up.put(rw.list_off.data(), rw.list_off.size()), at_lists = up.put(rw.lists.data(), rw.lists.size());
    const size_t at_words = up.put(s.words.data(), s.words.size());
    if (ws.alloc(s.workspace_bytes) != hipSuccess) {
        (void)hipGetLastError();
        return GRAB_OK;
    }
    GRAB_TRY(up.upload(base, &d_tab, st));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (kernel_ms) {
        GRAB_HIP(hipEventCreate(&e0));
        GRAB_HIP(hipEventCreate(&e1));
        GRAB_HIP(hipEventRecord(e0, st));
    }
    HalfScanArgs a{};
    a.data = d_dataset;
    a.queries = d_queries + (size_t)first * dim;
    a.row_query = d_tab.as<uint32_t>() + at_rq;
    a.row_lo = d_tab.as<uint32_t>() + at_lo;
    a.row_hi = d_tab.as<uint32_t>() + at_hi;
    a.list_off = d_tab.as<uint32_t>() + at_loff;
    a.lists = d_tab.as<uint32_t>() + at_lists;
    a.words = d_tab.as<uint32_t>() + at_words;
    a.out_ids = d_out_indices + (size_t)first * k;
    a.out_dist = d_out_dists + (size_t)first * k;
    a.contraction_done = e1;
    uint32_t* w = nullptr;
    float ms = 0.0f;
    int rc = half_scan_async(b, s, a, ws.ptr, num_cu, &w, st);
    uint32_t left[2] = {0, 0}, bad = 0;
    if (rc == GRAB_OK && hipMemcpyAsync(left, w, 8, hipMemcpyDeviceToHost, st) != hipSuccess) rc = GRAB_ERR_HIP;
    if (rc == GRAB_OK && !base && hipMemcpyAsync(&bad, b.scal + kScalBad, 4, hipMemcpyDeviceToHost, st) != hipSuccess) rc = GRAB_ERR_HIP;
    if (hipStreamSynchronize(st) != hipSuccess && rc == GRAB_OK) rc = GRAB_ERR_HIP;
    if (rc == GRAB_OK && kernel_ms && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = GRAB_ERR_HIP;
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (rc != GRAB_OK) {
        set_error("scan: the pass on f16 rows failed");
        return rc;
    }
    if (left[0] != 0 || bad != 0) return GRAB_OK;
    *applied = true;
    if (kernel_ms) *kernel_ms += ms;
    knn_stats().flop_f16 += rw.tiles * 2.0 * TM * TN * dim;
    knn_stats().flop_bf16 = 3.0 * knn_stats().flop_f16;
    if (left[1] == 0) return GRAB_OK;
    const SubRows own_rows = [&](const std::vector<uint32_t>& which, ScanRows* out) {
        std::vector<uint32_t> of_call(which);
        for (uint32_t& q : of_call) q += first;
        sub_rows(of_call, out);
    };
    // These are few as a rule, and the fp32 instructions' error is the smallest; halves of all rows are made for many
    const bool halves = left[1] >= kHalfPassQueries || (base && base->rows_split);
    return unproven_queries(d_dataset, num_dataset, dim, own_rows, a.queries, k, metric, w + 1, left[1], a.out_ids, a.out_dist, st, halves ? kAsHalves : kAsTheyAre,
                            halves ? base : nullptr);
}

// The f16 way.  *applied = false: nothing is to be used of it.
int scan_topk_half(const float* d_dataset, size_t num_dataset, uint32_t dim, const ScanRows& rw, const SubRows& sub_rows, const float* d_queries,
                   size_t num_queries, uint32_t k, int metric, int64_t* d_out_indices, float* d_out_dists, float* kernel_ms, hipStream_t st,
                   const ScanBase* base, uint32_t num_cu, bool* applied) {
    DeviceScratch base_mem;
    HalfBase own;
    *applied = false;
    if (!base) {
        if (base_mem.alloc(half_base_bytes(num_dataset, dim)) != hipSuccess) {
            (void)hipGetLastError();
            return GRAB_OK;
        }
        GRAB_TRY(half_base_async(d_dataset, num_dataset, dim, metric, base_mem.ptr, &own, st));
    }
    GRAB_TRY(scan_half_pass(base ? *base->half : own, d_dataset, num_dataset, rw, sub_rows, d_queries, 0, (uint32_t)num_queries, k, metric, d_out_indices, d_out_dists,
                            kernel_ms, st, base, num_cu, applied));
    if (*applied) return GRAB_OK;
    GRAB_HIP(hipStreamSynchronize(st));  // (the rows just made are freed)
    if (kernel_ms) *kernel_ms = 0.0f;
    knn_stats().flop_f16 = knn_stats().flop_bf16 = 0.0;
    knn_stats().exact_rows = 0;
    return GRAB_OK;
}

// The quick way.  One contraction over all tile-grid rows, which read their query's row in place; where there are
// fewer row tiles than workgroups a tile's sweep over its columns is cut into `splits` work items.  The lists of a
// query's rows - GEMM-form keys - are merged into one before anything is re-scored: the exact re-scoring and its
// check run once per query, not once per tile-grid row.  Queries that the check cannot prove go the plain way.
int scan_topk(const float* d_dataset, size_t num_dataset, uint32_t dim, const ScanRows& rw, const SubRows& sub_rows,
              const float* d_queries, size_t num_queries, uint32_t k, int metric, int64_t* d_out_indices, float* d_out_dists,
              float* kernel_ms, hipStream_t st, const ScanBase* base, RowsAs rows_as) {
    const uint32_t rows = rw.rows, nq = (uint32_t)num_queries;
    knn_stats().flop = knn_stats().flop_bf16 = knn_stats().flop_f16 = 0.0;
    knn_stats().redone_rows = knn_stats().exact_rows = 0;
    if (rows == 0) return no_row_admitted(num_queries, k, d_out_indices, d_out_dists, st);
    int dev = 0, num_cu = 0;
    GRAB_HIP(hipGetDevice(&dev));
    GRAB_HIP(hipDeviceGetAttribute(&num_cu, hipDeviceAttributeMultiprocessorCount, dev));
    const uint32_t kk = std::max<uint32_t>(2 * k + 32, 64);  // <= 288
    const uint32_t row_tiles = rows / TM, col_tiles = (uint32_t)((num_dataset + TN - 1) / TN), target = (uint32_t)num_cu * 2;
    // a prepared base has paid for its split rows; otherwise splitting a million rows pays from a thousand query rows on
    bool split = base ? base->split : rows_as != kAsTheyAre && knn_bf16_allowed() && dim % KC == 0 && rows >= 1024 && num_dataset >= 4096;
    // On f16 rows, except narrow intervals with short lists: a tenth of an interval's columns would be listed, and writing all values costs
    // less.  What this way saves goes with the products of the sweep, of which it takes one of three, with the queries, and with the
    // columns that one query's wave selects from; against that stand some 25 us of launches and of sampling.  Seven row sets from 300,000 x 32 to
    // 150,000 x 768, 1 to 10,000 queries, intervals of 3000 to 15,000, k 10 and 16, a call over a prepared base: the rule's choice takes
    // 0.3 % more than the better one in the mean, 4 % more than stored values at worst (a line at 6000 columns: 2 %, and 19 %).  Intervals of
    // 3000, 6000 and 11,000, k 10, stored values against this way in us:
    //   300,000 x 32   1 query 69 / 84, 76 / 85, 86 / 86;         300 106 / 131, 113 / 132, 126 / 131;   10,000 273 / 285, 343 / 300, 458 / 320
    //   1M x 128       1       73 / 93, 81 / 87, 92 / 92;         300 240 / 230, 250 / 221, 265 / 213;   10,000 443 / 398, 529 / 409, 666 / 428
    //   150,000 x 768  1       101 / 111, 115 / 110, 128 / 114;   300 216 / 207, 228 / 195, 242 / 191;   10,000 579 / 437, 735 / 494, 1027 / 585
    // Below 3000 none was measured to gain (1000, 10,000 queries of 1M x 128: 384 / 582).  Longer lists, selection inside the contraction against
    // this: k 40, 10,000 queries, 1000 columns 1361 / 472, 20,000 3743 / 574.
    bool narrow = false;
    if (rw.one_row_per_query && kk <= 64) {
        const double queries = (double)rw.lists.size(), mean = (double)rw.columns / queries;
        narrow = mean < 3000.0 || rw.tiles * dim / 30000.0 + queries / 800.0 + mean / 430.0 < 26.0;
    }
    // Beyond 127,000 columns a sampled value stands for more than 64 columns, too few lie within a bound to set it by; by the same
    // reckoning as at 100,000 from one in 130 (scan_half.hip: 5.3 ms a call against 3.3 with stored values).
    bool on_half = rows_as == kOnF16 && split && half_scan_takes(rw.widest) && (!base || base->half), applied = false;
    if (on_half && !rw.one_row_per_query) {
        uint32_t most = 0;  // rows of a query; a wave's lanes hold them
        for (size_t q = 0; q < num_queries; ++q) most = std::max(most, rw.list_off[q + 1] - rw.list_off[q]);
        on_half = most <= 64;
    }
    auto run_half = [&] {
        return scan_topk_half(d_dataset, num_dataset, dim, rw, sub_rows, d_queries, num_queries, k, metric, d_out_indices, d_out_dists, kernel_ms, st, base,
                              (uint32_t)num_cu, &applied);
    };
    if (on_half && !narrow) {
        GRAB_TRY(run_half());
        if (applied) return GRAB_OK;
    }
    if (base && base->split && base->rows_split == nullptr) {
        bool no_room = false;
        GRAB_TRY(base->make_split(st, &no_room));
        if (no_room) {  // the halves do not fit beside the f16 rows: these serve narrow intervals as well, the rows as they are what is left
            if (on_half && narrow) GRAB_TRY(run_half());
            if (applied) return GRAB_OK;
            base = nullptr;
            split = false;
        }
    }
    DeviceScratch d_tab, buf, cand, merged, outside, norm_a, norm_b, split_a, split_b, mean, doubt;
    // Short candidate lists (k <= 16) go the dense way: the contraction writes the distances of the columns that a row tile
    // sweeps, in work items of equal length, and a streaming pass keeps the kk smallest of every row.  The other way
    // selects inside the contraction: its thresholds start open for every row and tighten over the first hundreds of
    // admitted columns - most of a narrow interval, and again in every item that a long sweep is cut into, so sweeps are
    // cut only until every workgroup has an item and the longest one sets the time.  4999 queries with 1-4 of 64 buckets
    // on 200k x 768 (mean sweep 23 column tiles, longest 128): 2.70 -> 0.35 ms of contraction, 0.08 ms of selection.  In
    // passes of at most 128 row tiles whose distances fit a bound: for buckets what the buffers of the other way would take.
    const uint64_t dense_cap = rw.one_row_per_query ? 4ull << 30 : (uint64_t)target * TM * CAP * sizeof(uint64_t);
    constexpr uint64_t kTileBytes = (uint64_t)TM * TN * sizeof(float);
    struct Pass {
        uint32_t t0, t1;
    };
    std::vector<Pass> passes;
    uint64_t dense_bytes = 0;
    bool dense_way = kk <= 64;
    for (uint32_t t0 = 0; t0 < row_tiles && dense_way;) {
        uint32_t t1 = t0;
        uint64_t bytes = 0;
        while (t1 < row_tiles && t1 - t0 < 128) {
            const uint64_t more = (rw.tile_hi[t1] - rw.tile_lo[t1]) * kTileBytes;
            if (bytes + more > dense_cap) break;
            bytes += more;
            ++t1;
        }
        if (t1 == t0) dense_way = false;  // one row tile's sweep alone is beyond the cap
        dense_bytes = std::max(dense_bytes, bytes);
        passes.push_back({t0, t1});
        t0 = t1;
    }
    // enough work items for every workgroup of the grid, and no more: an item ends with a selection over each of its
    // 128 rows, which costs as much as several tile steps (1M x 768, 10,000 queries: 2 splits 6.9 ms, 5 splits 8.2 ms)
    const uint32_t splits = dense_way ? 1u : std::max(1u, std::min({(target + row_tiles - 1) / row_tiles, 8u, 1024u / kk}));
    const uint32_t grid = std::min(row_tiles * splits, target);
    const bool per_query = dense_way && rw.one_row_per_query;  // the selection leaves a query's list, nothing to merge
    if (!dense_way) GRAB_HIP(buf.alloc((size_t)grid * TM * CAP * sizeof(uint64_t)));
    if (!per_query) GRAB_HIP(cand.alloc((size_t)rows * splits * kk * sizeof(uint64_t)));
    GRAB_HIP(merged.alloc((size_t)nq * kk * sizeof(uint64_t)));
    GRAB_HIP(outside.alloc((size_t)nq * 4));
    GRAB_HIP(norm_a.alloc((size_t)nq * 4));
    if (!base) GRAB_HIP(norm_b.alloc(num_dataset * 4));
    // [0] rows not proven, [1..nq] which, [nq+1] max norm of the base rows, from [nq+3] a work counter per launch
    const uint32_t n_counters = (uint32_t)std::min<size_t>(passes.size() + 1, 256);
    GRAB_HIP(doubt.alloc(((size_t)nq + 3 + n_counters) * 4));
    // the host's tables: per tile-grid row its query and column range, per query its rows, per pass its work list
    ScanUpload up;
    up.tab.reserve((size_t)rows * 3 + rw.list_off.size() + rw.lists.size() + passes.size() * kSchedWords + 64);
    const size_t at_rq = up.put(rw.row_query.data(), rows), at_lo = up.put(rw.row_lo.data(), rows), at_hi = up.put(rw.row_hi.data(), rows);
    const size_t at_loff = up.put(rw.list_off.data(), rw.list_off.size()), at_lists = up.put(rw.lists.data(), rw.lists.size());
    size_t at_sched = 0;
    if (dense_way) {
        std::vector<uint32_t> sched(passes.size() * (size_t)kSchedWords, 0u);
        for (size_t pi = 0; pi < passes.size(); ++pi) {
            const Pass& ps = passes[pi];
            dense_sched(rw.tile_lo.data() + ps.t0, rw.tile_hi.data() + ps.t0, ps.t1 - ps.t0, target, sched.data() + pi * kSchedWords);
        }
        at_sched = up.put(sched.data(), sched.size());
    }
    GRAB_TRY(up.upload(base, &d_tab, st));
    const uint32_t* d_rq = d_tab.as<uint32_t>() + at_rq;
    const uint32_t* d_lo = d_tab.as<uint32_t>() + at_lo;
    const uint32_t* d_hi = d_tab.as<uint32_t>() + at_hi;
    const uint32_t* d_loff = d_tab.as<uint32_t>() + at_loff;
    const uint32_t* d_lists = d_tab.as<uint32_t>() + at_lists;
    const uint32_t* d_sched_all = d_tab.as<uint32_t>() + at_sched;
    {
        const size_t fill = per_query ? (size_t)nq * kk : 0;  // a query without a row keeps an empty list
        hipLaunchKernelGGL(scan_init_kernel, dim3((uint32_t)std::min<size_t>(std::max<size_t>((fill + 255) / 256, 1), 1024)), dim3(256), 0, st,
                           doubt.as<uint32_t>(), nq, n_counters, merged.as<uint64_t>(), fill);
        GRAB_HIP(hipGetLastError());
    }
    TileArgs t{};
    t.A = d_queries;
    t.B = d_dataset;
    const float* d_norm_b = base ? base->norm : norm_b.as<float>();
    const float* d_max_norm_b = base ? base->max_norm : reinterpret_cast<const float*>(doubt.as<uint32_t>() + nq + 1);
    if (split) {
        // rows as bf16 halves (centred on the base's mean for squared L2); their norms serve the distance form and the
        // error bound of the check alike
        GRAB_HIP(split_a.alloc((size_t)nq * dim * 4));
        const float* mu = base ? base->mean : nullptr;
        if (!base) {
            GRAB_HIP(split_b.alloc(num_dataset * dim * 4));
            GRAB_TRY(split_base_rows(d_dataset, num_dataset, dim, metric, &mean, split_b.as<uint16_t>(), norm_b.as<float>(), st));
            mu = mean.as<float>();
        }
        launch_split_rows_chunked(d_queries, nq, dim, mu, split_a.as<uint16_t>(), norm_a.as<float>(), st);
        t.A = split_a.as<float>();
        t.B = base ? reinterpret_cast<const float*>(base->rows_split) : split_b.as<float>();
    } else {
        if (!base) launch_row_norms(d_dataset, num_dataset, dim, norm_b.as<float>(), st);
        launch_row_norms(d_queries, nq, dim, norm_a.as<float>(), st);
    }
    if (!base) launch_max_float(norm_b.as<float>(), num_dataset, doubt.as<uint32_t>() + nq + 1, st);
    GRAB_HIP(hipGetLastError());
    t.normA = norm_a.as<float>();
    t.normB = d_norm_b;
    t.row_perm = d_rq;
    t.row_lo = d_lo;
    t.row_hi = d_hi;
    t.range_by_grid_row = 1;
    t.cand_by_grid_row = 1;
    t.buf = buf.as<uint64_t>();
    t.cand_out = cand.as<uint64_t>();
    t.M = rows;
    t.N = (uint32_t)num_dataset;
    t.dim = dim;
    t.kk = kk;
    t.nsplit = splits;
    t.col_tiles = col_tiles;
    t.tiles_per_split = (col_tiles + splits - 1) / splits;
    t.row_tiles = row_tiles;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (kernel_ms) {
        GRAB_HIP(hipEventCreate(&e0));
        GRAB_HIP(hipEventCreate(&e1));
        GRAB_HIP(hipEventRecord(e0, st));
    }
    int rc = GRAB_OK;
    DeviceScratch dense;
    if (dense_way) {
        if (dense.alloc(dense_bytes) != hipSuccess) {
            set_error("scan: out of device memory for %llu bytes of distances", (unsigned long long)dense_bytes);
            rc = GRAB_ERR_HIP;
        }
        for (size_t pi = 0; pi < passes.size() && rc == GRAB_OK; ++pi) {
            const Pass& ps = passes[pi];
            TileArgs tp = t;
            tp.row_perm = d_rq + (size_t)ps.t0 * TM;
            tp.row_lo = d_lo + (size_t)ps.t0 * TM;
            tp.row_hi = d_hi + (size_t)ps.t0 * TM;
            tp.M = (ps.t1 - ps.t0) * TM;
            tp.row_tiles = ps.t1 - ps.t0;
            tp.nsplit = 1;
            tp.dense = dense.as<float>();
            tp.dense_rel = 1;
            tp.sched = d_sched_all + pi * kSchedWords;
            tp.work_counter = pi < n_counters ? doubt.as<uint32_t>() + nq + 3 + pi : nullptr;
            rc = launch_tile_store(tp, metric, target, st, split);
            if (rc != GRAB_OK) break;
            hipLaunchKernelGGL(stream_select_keys_kernel, dim3((tp.M + 3) / 4), dim3(256), 0, st, dense.as<float>(),
                               per_query ? tp.row_perm : nullptr, tp.row_lo, tp.row_hi, tp.sched, tp.M, kk,
                               per_query ? merged.as<uint64_t>() : cand.as<uint64_t>() + (size_t)ps.t0 * TM * kk);
            if (hipGetLastError() != hipSuccess) {
                set_error("scan: select kernel launch failed");
                rc = GRAB_ERR_HIP;
            }
        }
    } else {
        t.work_counter = doubt.as<uint32_t>() + nq + 3;
        rc = launch_tile_any(t, metric, kFilterColRange, grid, st, split);
    }
    if (kernel_ms && rc == GRAB_OK) {
        hipError_t e = hipEventRecord(e1, st);
        if (e == hipSuccess) e = hipEventSynchronize(e1);
        if (e == hipSuccess) e = hipEventElapsedTime(kernel_ms, e0, e1);
        if (e != hipSuccess) {
            set_error("HIP error %s while timing the contraction kernel", hipGetErrorString(e));
            rc = GRAB_ERR_HIP;
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (rc != GRAB_OK) {
        (void)hipStreamSynchronize(st);  // the host tables and the scratch above go out of scope
        return rc;
    }
    const double flop = rw.tiles * 2.0 * TM * TN * dim;
    if (split) knn_stats().flop_bf16 = 3.0 * flop;  // three instructions a product
    else knn_stats().flop = flop;
    if (!per_query)
        hipLaunchKernelGGL(premerge_lists_kernel, dim3((nq + 3) / 4), dim3(256), 0, st, cand.as<uint64_t>(), splits, kk, d_loff, d_lists, nq,
                           merged.as<uint64_t>(), outside.as<float>());
    RefineArgs r{};
    r.A = d_queries;
    r.B = d_dataset;
    r.cand = merged.as<uint64_t>();
    r.out_i64 = d_out_indices;
    r.out_dist = d_out_dists;
    r.M = nq;
    r.dim = dim;
    r.nc = kk;
    r.k = k;
    r.kk = kk;
    r.normA = norm_a.as<float>();
    r.max_normB = d_max_norm_b;
    r.sorted = 1;
    r.outside_in = per_query ? nullptr : outside.as<float>();  // one whole list per query: its last key is the bound
    r.doubt = doubt.as<uint32_t>();
    if (split) {
        r.split_normA = norm_a.as<float>();
        r.split_max_normB = r.max_normB;
        r.split_terms = 3.0f * (float)dim;
    }
    rc = launch_refine_any(r, metric, st);
    uint32_t n_doubt = 0;
    if (rc == GRAB_OK && hipMemcpyAsync(&n_doubt, doubt.ptr, 4, hipMemcpyDeviceToHost, st) != hipSuccess) rc = GRAB_ERR_HIP;
    if (hipStreamSynchronize(st) != hipSuccess && rc == GRAB_OK) rc = GRAB_ERR_HIP;
    if (rc != GRAB_OK) {
        set_error("scan: re-scoring failed");
        return rc;
    }
    if (n_doubt == 0) return GRAB_OK;
    return unproven_queries(d_dataset, num_dataset, dim, sub_rows, d_queries, k, metric, doubt.as<uint32_t>(), n_doubt, d_out_indices, d_out_dists, st);
}

}  // namespace
}  // namespace grab

using namespace grab;

extern "C" {

int grab_bucket_scan_topk(const float* d_dataset, size_t num_dataset, uint32_t dim, const uint64_t* h_bucket_offsets,
                          uint32_t num_buckets, const float* d_queries, size_t num_queries, uint32_t k, int metric,
                          const uint64_t* h_masks, int64_t* d_out_indices, float* d_out_dists, float* kernel_ms, void* stream) {
    GRAB_REQUIRE(d_dataset && d_queries && h_bucket_offsets && h_masks && d_out_indices && d_out_dists, "null pointer");
    GRAB_REQUIRE(num_buckets >= 1 && num_buckets <= 64, "num_buckets must be in [1,64] (a query's buckets are a 64-bit set)");
    GRAB_REQUIRE(k >= 1 && k <= 128, "k must be in [1,128]");
    GRAB_REQUIRE(dim >= 4 && dim % 4 == 0, "unsupported dimension %u (must be a multiple of 4)", dim);
    GRAB_REQUIRE(metric == kMetricL2 || metric == kMetricIP, "bad metric");
    GRAB_REQUIRE(num_dataset > 0 && num_dataset < (1ull << 31) && num_queries < (1ull << 31), "bad problem size");
    for (uint32_t b = 0; b < num_buckets; ++b)
        GRAB_REQUIRE(h_bucket_offsets[b] <= h_bucket_offsets[b + 1], "bucket offsets must not decrease");
    GRAB_REQUIRE(h_bucket_offsets[num_buckets] <= num_dataset, "the last bucket ends beyond the dataset");
    if (kernel_ms) *kernel_ms = 0.0f;
    if (num_queries == 0) return GRAB_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    ScanRows rw;
    scan_rows(h_bucket_offsets, num_buckets, h_masks, num_queries, &rw);
    const SubRows sub_rows = [&](const std::vector<uint32_t>& which, ScanRows* out) {
        std::vector<uint64_t> sub_masks(which.size());
        for (size_t i = 0; i < which.size(); ++i) sub_masks[i] = h_masks[which[i]];
        scan_rows(h_bucket_offsets, num_buckets, sub_masks.data(), which.size(), out);
    };
    return scan_topk(d_dataset, num_dataset, dim, rw, sub_rows, d_queries, num_queries, k, metric, d_out_indices, d_out_dists, kernel_ms, st, nullptr, kOnF16);
}

int grab_window_scan_topk(const float* d_dataset, size_t num_dataset, uint32_t dim, const float* d_queries, size_t num_queries,
                          uint32_t k, int metric, const uint64_t* h_id_lo, const uint64_t* h_id_hi, int64_t* d_out_indices,
                          float* d_out_dists, float* kernel_ms, void* stream) {
    GRAB_REQUIRE(d_dataset && d_queries && h_id_lo && h_id_hi && d_out_indices && d_out_dists, "null pointer");
    GRAB_REQUIRE(k >= 1 && k <= 128, "k must be in [1,128]");
    GRAB_REQUIRE(dim >= 4 && dim % 4 == 0, "unsupported dimension %u (must be a multiple of 4)", dim);
    GRAB_REQUIRE(metric == kMetricL2 || metric == kMetricIP, "bad metric");
    GRAB_REQUIRE(num_dataset > 0 && num_dataset < (1ull << 31) && num_queries < (1ull << 31), "bad problem size");
    if (kernel_ms) *kernel_ms = 0.0f;
    if (num_queries == 0) return GRAB_OK;
    ScanRows rw;
    window_rows(h_id_lo, h_id_hi, nullptr, num_queries, num_dataset, &rw);
    const SubRows sub_rows = [&](const std::vector<uint32_t>& which, ScanRows* out) {
        window_rows(h_id_lo, h_id_hi, which.data(), which.size(), num_dataset, out);
    };
    return scan_topk(d_dataset, num_dataset, dim, rw, sub_rows, d_queries, num_queries, k, metric, d_out_indices, d_out_dists, kernel_ms,
                     static_cast<hipStream_t>(stream), nullptr, kOnF16);
}

// A base prepared for the two scans: what a call would otherwise make of the base rows every time, and a block of
// device memory that the calls' scratch is taken from.
struct grab_scan_base {
    const float* d_dataset = nullptr;
    size_t num_dataset = 0;
    uint32_t dim = 0;
    int metric = 0;
    DeviceScratch rows_split, norm, mean, max_norm, half_mem;
    HalfBase half;
    ScanBase view;
    void* block = nullptr;  // scratch of the calls; grown to what the last call asked for
    size_t block_bytes = 0;
    void* staging = nullptr;  // page-locked host memory for a call's tables
    size_t staging_bytes = 0;
};

int grab_scan_base_create(const float* d_dataset, size_t num_dataset, uint32_t dim, int metric, grab_scan_base** out) {
    GRAB_REQUIRE(d_dataset && out, "null pointer");
    GRAB_REQUIRE(dim >= 4 && dim % 4 == 0, "unsupported dimension %u (must be a multiple of 4)", dim);
    GRAB_REQUIRE(metric == kMetricL2 || metric == kMetricIP, "bad metric");
    GRAB_REQUIRE(num_dataset > 0 && num_dataset < (1ull << 31), "bad problem size");
    auto* b = new grab_scan_base();
    b->d_dataset = d_dataset;
    b->num_dataset = num_dataset;
    b->dim = dim;
    b->metric = metric;
    auto fail = [&](int rc) {
        grab_scan_base_destroy(b);
        return rc;
    };
    b->view.split = knn_bf16_allowed() && dim % KC == 0 && num_dataset >= 4096;
    if (b->view.split) {
        // f16 rows are what the calls use first; rows as bf16 halves are made when one needs them - at once where a row is not finite, or
        // all point one way
        uint32_t found[kScalOneWay + 1] = {};
        if (b->half_mem.alloc(half_base_bytes(num_dataset, dim)) != hipSuccess) {
            (void)hipGetLastError();
            set_error("scan base: out of device memory");
            return fail(GRAB_ERR_HIP);
        }
        const int rc = half_base_async(d_dataset, num_dataset, dim, metric, b->half_mem.ptr, &b->half, nullptr);
        if (rc != GRAB_OK) return fail(rc);
        if (hipMemcpy(found, b->half.scal, sizeof(found), hipMemcpyDeviceToHost) != hipSuccess) {
            set_error("scan base: preparing the rows failed");
            return fail(GRAB_ERR_HIP);
        }
        if (found[kScalBad] == 0 && found[kScalOneWay] == 0) {
            b->view.half = &b->half;
        } else {
            (void)hipFree(b->half_mem.ptr);
            b->half_mem.ptr = nullptr;
        }
    }
    // norms, and the rows as bf16 halves: now for a base that is scanned as it is, or when a call first needs them
    auto prepare = [b](hipStream_t st, bool* no_room) -> int {
        DeviceScratch norm, max_norm, mean, rows_split;  // the base's once all is queued
        ScratchArena* const lent = scratch_arena();
        scratch_arena() = nullptr;  // these stay: no part of a call's scratch
        *no_room = norm.alloc(b->num_dataset * 4) != hipSuccess || max_norm.alloc(4) != hipSuccess ||
                   (b->view.split && rows_split.alloc(b->num_dataset * b->dim * 4) != hipSuccess);
        int rc = GRAB_OK;
        if (*no_room) (void)hipGetLastError();
        else if (b->view.split) rc = split_base_rows(b->d_dataset, b->num_dataset, b->dim, b->metric, &mean, rows_split.as<uint16_t>(), norm.as<float>(), st);
        else launch_row_norms(b->d_dataset, b->num_dataset, b->dim, norm.as<float>(), st);
        scratch_arena() = lent;
        if (rc != GRAB_OK || *no_room) return rc;
        GRAB_HIP(hipMemsetAsync(max_norm.ptr, 0, 4, st));
        launch_max_float(norm.as<float>(), b->num_dataset, max_norm.as<uint32_t>(), st);
        GRAB_HIP(hipGetLastError());
        std::swap(b->norm.ptr, norm.ptr);
        std::swap(b->max_norm.ptr, max_norm.ptr);
        std::swap(b->mean.ptr, mean.ptr);
        std::swap(b->rows_split.ptr, rows_split.ptr);
        b->view.rows_split = b->rows_split.as<uint16_t>();
        b->view.norm = b->norm.as<float>();
        b->view.mean = b->mean.as<float>();
        b->view.max_norm = b->max_norm.as<float>();
        return GRAB_OK;
    };
    b->view.make_split = prepare;
    if (b->view.half == nullptr) {
        bool no_room = false;
        const int rc = prepare(nullptr, &no_room);
        if (no_room) {
            set_error("scan base: out of device memory");
            return fail(GRAB_ERR_HIP);
        }
        if (rc != GRAB_OK) return fail(rc);
    }
    if (hipDeviceSynchronize() != hipSuccess) {
        set_error("scan base: preparing the rows failed");
        return fail(GRAB_ERR_HIP);
    }
    b->view.staging = &b->staging;
    b->view.staging_bytes = &b->staging_bytes;
    *out = b;
    return GRAB_OK;
}

void grab_scan_base_destroy(grab_scan_base* b) {
    if (!b) return;
    if (b->block) (void)hipFree(b->block);
    if (b->staging) (void)hipHostFree(b->staging);
    delete b;
}

namespace {
// a scan with the calls' scratch taken from the base's block; the block follows what the call asked for (up to 8 GiB:
// beyond that, and on the first call, scratch is allocated as ever)
int scan_on_base(grab_scan_base* b, const std::function<int()>& run) {
    ScratchArena arena{static_cast<char*>(b->block), b->block_bytes, 0, 0};
    struct Lend {  // the calling thread's scratch comes from the block until this scope ends, however it ends
        ScratchArena*& slot;
        ScratchArena* const before;
        Lend(ScratchArena* a) : slot(scratch_arena()), before(slot) { slot = a; }
        ~Lend() { slot = before; }
    };
    int rc;
    {
        Lend lend(&arena);
        rc = run();  // returns with the stream drained: nothing of the block is in use any more
    }
    if (rc != GRAB_OK) (void)hipDeviceSynchronize();  // a call that gave up half way may have left kernels queued
    const size_t most = std::max(arena.wanted, arena.peak), want = std::min<size_t>(most + most / 8 + (1u << 20), 8ull << 30);
    if (most > b->block_bytes && want > b->block_bytes) {
        if (b->block) (void)hipFree(b->block);
        b->block = nullptr;
        b->block_bytes = 0;
        if (hipMalloc(&b->block, want) == hipSuccess) b->block_bytes = want;
        else (void)hipGetLastError();  // no block: the next call allocates as this one did
    }
    return rc;
}
}  // namespace

int grab_scan_base_window_topk(grab_scan_base* b, const float* d_queries, size_t num_queries, uint32_t k, const uint64_t* h_id_lo,
                               const uint64_t* h_id_hi, int64_t* d_out_indices, float* d_out_dists, float* kernel_ms, void* stream) {
    GRAB_REQUIRE(b && d_queries && h_id_lo && h_id_hi && d_out_indices && d_out_dists, "null pointer");
    GRAB_REQUIRE(k >= 1 && k <= 128, "k must be in [1,128]");
    GRAB_REQUIRE(num_queries < (1ull << 31), "bad problem size");
    if (kernel_ms) *kernel_ms = 0.0f;
    if (num_queries == 0) return GRAB_OK;
    ScanRows rw;
    window_rows(h_id_lo, h_id_hi, nullptr, num_queries, b->num_dataset, &rw);
    const SubRows sub_rows = [&](const std::vector<uint32_t>& which, ScanRows* out) {
        window_rows(h_id_lo, h_id_hi, which.data(), which.size(), b->num_dataset, out);
    };
    return scan_on_base(b, [&]() {
        return scan_topk(b->d_dataset, b->num_dataset, b->dim, rw, sub_rows, d_queries, num_queries, k, b->metric, d_out_indices,
                         d_out_dists, kernel_ms, static_cast<hipStream_t>(stream), &b->view, kOnF16);
    });
}

int grab_scan_base_bucket_topk(grab_scan_base* b, const uint64_t* h_bucket_offsets, uint32_t num_buckets, const float* d_queries,
                               size_t num_queries, uint32_t k, const uint64_t* h_masks, int64_t* d_out_indices, float* d_out_dists,
                               float* kernel_ms, void* stream) {
    GRAB_REQUIRE(b && d_queries && h_bucket_offsets && h_masks && d_out_indices && d_out_dists, "null pointer");
    GRAB_REQUIRE(num_buckets >= 1 && num_buckets <= 64, "num_buckets must be in [1,64] (a query's buckets are a 64-bit set)");
    GRAB_REQUIRE(k >= 1 && k <= 128, "k must be in [1,128]");
    GRAB_REQUIRE(num_queries < (1ull << 31), "bad problem size");
    for (uint32_t i = 0; i < num_buckets; ++i)
        GRAB_REQUIRE(h_bucket_offsets[i] <= h_bucket_offsets[i + 1], "bucket offsets must not decrease");
    GRAB_REQUIRE(h_bucket_offsets[num_buckets] <= b->num_dataset, "the last bucket ends beyond the dataset");
    if (kernel_ms) *kernel_ms = 0.0f;
    if (num_queries == 0) return GRAB_OK;
    ScanRows rw;
    scan_rows(h_bucket_offsets, num_buckets, h_masks, num_queries, &rw);
    const SubRows sub_rows = [&](const std::vector<uint32_t>& which, ScanRows* out) {
        std::vector<uint64_t> sub_masks(which.size());
        for (size_t i = 0; i < which.size(); ++i) sub_masks[i] = h_masks[which[i]];
        scan_rows(h_bucket_offsets, num_buckets, sub_masks.data(), which.size(), out);
    };
    return scan_on_base(b, [&]() {
        return scan_topk(b->d_dataset, b->num_dataset, b->dim, rw, sub_rows, d_queries, num_queries, k, b->metric, d_out_indices,
                         d_out_dists, kernel_ms, static_cast<hipStream_t>(stream), &b->view, kOnF16);
    });
}

}  // extern "C"
