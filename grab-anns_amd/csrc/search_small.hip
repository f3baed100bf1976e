// Beam search over the CAGRA graph for small batches: one workgroup of 1024 or 512 threads per query.
//
// Same algorithm and same results as search.hip (the loop of the reference's search_kernel / search_kernel_bucket /
// search_kernel_range, src/index/search.cu:149-370, :375-586, :589-798), arranged for the time that ONE query takes:
// with fewer queries than the device has room for, that is the time of the call.  A query is a chain of 15 - 45
// iterations on one CU; an iteration costs trips to LDS, two trips to the second-level cache or beyond - and the
// vector instructions of its waves: a wave's instruction keeps a SIMD for four cycles, so sixteen waves that go through
// a hundred instructions each are 1600 cycles, however short each wave's own chain is.  Hence no more waves in a phase
// than it has work for, and phases with one barrier behind each:
//   1. pick the parents: the first unexpanded entries of the queue and the candidates, ranked among each other;
//   2. some waves read the parents' graph rows, one neighbour a lane: visited set, filter, survivor list - while others
//      merge the candidates into the queue;
//   3. score the survivors, 8 lanes a row, all waves; those that beat the worst entry are the next candidates.
// What bounds it: the chain.  An iteration takes about 7000 cycles at itopk 256 and 5500 at 128, of which the two trips to
// memory are 700 and 900 - 1800 (146 survivors of 512 bytes go through one CU); the rest is ten trips to LDS and some 500
// instructions.  Against the 1024-thread kernel with five barriers and a merge of its own before the expansion: one query
// on 100k x 128, itopk 256, width 6, 44 iterations: 207 -> 140 us; 100 queries with a shared window on 200k x 96, itopk
// 128: 166 -> 101 us; 64 rows of an insert into 200k x 128, itopk 128, width 6: 90 -> 70 us.
// Tried and left out: scoring each wave's own survivors without the hand-over (16 waves that each go through the whole
// expansion: 184 us); a wave per candidate, and sixteen queue entries a wave with four lanes each, in the merge (168 and
// 157 us: more instructions); touching the graph row of every candidate ahead of time (the registers that wait for the
// words are moved between branches, which waits for them: 160 us with and without).
#include "search_internal.hpp"

namespace grab {

using namespace dev;

namespace {

// M_NCAND: two counters used in turn - while the candidates of one are merged the other one counts the next ones.  The
// same goes for the two lists of unexpanded entries.
enum { M_NCAND = 0, M_NSURV = 2, M_TAIL, M_PAR, M_F, M_FULL, M_USED, M_COUNT };

struct Lds {
    float* query;
    uint64_t* top;   // two queues, `padded` places each: one is merged into the other
    uint16_t* open;  // two lists: unexpanded entries before each queue place
    uint32_t padded;
    uint64_t* ahead;  // two lists: the first search_width unexpanded queue entries
    uint64_t* cand;
    uint64_t* marked;  // places of the merged queue that candidates take, a bit each
    uint32_t* surv;
    uint32_t* parents;
    uint32_t* misc;
    uint32_t* table;
};

__device__ __forceinline__ Lds carve(uint8_t* smem, const SearchArgs& a) {
    const SearchSmallLdsLayout lay = search_small_lds_layout(a.itopk, a.dim, a.cmax, a.search_width, a.table_bitlen);
    Lds l;
    l.query = reinterpret_cast<float*>(smem + lay.off_query);
    l.padded = search_small_padded_queue(a.itopk);
    l.top = reinterpret_cast<uint64_t*>(smem + lay.off_top);
    l.open = reinterpret_cast<uint16_t*>(smem + lay.off_open);
    l.ahead = reinterpret_cast<uint64_t*>(smem + lay.off_ahead);
    l.cand = reinterpret_cast<uint64_t*>(smem + lay.off_cand);
    l.marked = reinterpret_cast<uint64_t*>(smem + lay.off_marked);
    l.surv = reinterpret_cast<uint32_t*>(smem + lay.off_surv);
    l.parents = reinterpret_cast<uint32_t*>(smem + lay.off_parents);
    l.misc = reinterpret_cast<uint32_t*>(smem + lay.off_misc);
    l.table = reinterpret_cast<uint32_t*>(smem + lay.off_hash);
    return l;
}

template <int FILTER>
struct FilterState {
    uint64_t start, end, mask;
};

template <int FILTER>
__device__ __forceinline__ bool filter_pass(const SearchArgs& a, const FilterState<FILTER>& f, uint32_t id) {
    if (FILTER == kFilterRange) {
        const uint64_t t = a.ts[id];
        return t >= f.start && t < f.end;  // [start,end), compute_distance.cuh:580-584
    }
    if (FILTER == kFilterMask) return (f.mask >> (a.labels[id] & 63)) & 1ull;
    if (FILTER == kFilterIdRange) return id >= f.start && id < f.end;  // nothing to read
    if (FILTER == kFilterRank) {
        const uint64_t x = a.rank_of_id[id];  // the row's place in timestamp order
        return x >= f.start && x < f.end;
    }
    return true;
}

// Reserves a place in a list for the lane.  The lanes' additions meet at one address and are answered one after the other
// (16 of them in about 80 cycles); collected in one lane first they would take twice that, most of it the branch and the
// hand-out.  The address is made to look different from lane to lane, which keeps the compiler from collecting them.
__device__ __forceinline__ uint32_t lds_append(uint32_t* length) {
    asm volatile("" : "+v"(length));
    return __hip_atomic_fetch_add((__attribute__((address_space(3))) uint32_t*)length, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Scores the survivors s0 .. s0 + 7 of the list (one row per group of 8 lanes; with TWO the rows `next` places further
// on as well, so that twice as many loads are in flight) and appends those that beat `worst` to the candidate list.
template <int CPL, int METRIC, bool TWO>
__device__ __forceinline__ void score_round(const SearchArgs& a, const Lds& l, const float4 (&qreg)[CPL ? CPL : 1], uint32_t ns,
                                            uint32_t s0, uint32_t next, uint64_t worst, uint32_t* ncand, int lane) {
    const int grp = lane >> 3, j = lane & 7;
    const uint32_t sa = s0 + grp, sb = sa + next;
    uint64_t k0 = kInvalidKey, k1 = kInvalidKey;
    if (sa < ns) {
        const bool two = TWO && sb < ns;
        const uint32_t id0 = l.surv[sa];
        const uint32_t id1 = two ? l.surv[sb] : id0;
        const float4* r0 = reinterpret_cast<const float4*>(a.data + (size_t)id0 * a.dim);
        const float4* r1 = reinterpret_cast<const float4*>(a.data + (size_t)id1 * a.dim);
        float d0 = 0.0f, d1 = 0.0f;
        if (CPL > 0) {
            float4 v0[CPL ? CPL : 1], v1[CPL ? CPL : 1];
#pragma unroll
            for (int c = 0; c < CPL; ++c) v0[c] = r0[c * 8 + j];
            if (TWO) {
#pragma unroll
                for (int c = 0; c < CPL; ++c) v1[c] = r1[c * 8 + j];
            }
#pragma unroll
            for (int c = 0; c < CPL; ++c) d0 = fold4<METRIC>(d0, qreg[c], v0[c]);
            if (TWO) {
#pragma unroll
                for (int c = 0; c < CPL; ++c) d1 = fold4<METRIC>(d1, qreg[c], v1[c]);
            }
        } else {
            fold_rows_any<METRIC, TWO>(r0, r1, reinterpret_cast<const float4*>(l.query), j, a.dim >> 2, d0, d1);
        }
        d0 = group8_sum(d0);
        k0 = make_key(METRIC == kMetricIP ? -d0 : d0, id0);
        if (TWO) {
            d1 = group8_sum(d1);
            if (two) k1 = make_key(METRIC == kMetricIP ? -d1 : d1, id1);
        }
    }
    const bool p0 = (j == 0) & (k0 < worst), p1 = TWO && ((j == 0) & (k1 < worst));
    if (p0) l.cand[lds_append(ncand)] = k0;
    if (p1) l.cand[lds_append(ncand)] = k1;
}

// The merge of the candidate list into the sorted queue.  An entry's new position is the number of entries ordered
// before it by (distance,id); the expanded flag takes no part in the order and queue entries go ahead of equal
// candidates.  The parents are the first search_width unexpanded entries of the merged queue
// (src/index/search.cu:38-107): `open` holds for every queue place how many unexpanded entries lie before it, with the
// candidates (never expanded) ahead of an entry that is its place among the unexpanded ones, and the first of them get
// their flag set - so every count of the merged queue is that much smaller, and the entries next in line make the list
// of the first unexpanded entries that the next pick starts from.
struct Merge {
    const uint64_t* src;
    uint64_t* dst;
    const uint16_t* open_src;
    uint16_t* open_dst;
    uint32_t width;
    uint32_t* parents;  // null: picked already
    uint64_t* next;     // the first unexpanded entries of the merged queue
    __device__ __forceinline__ void place(uint64_t k, uint32_t r, uint32_t before, bool unexpanded) const {  // before: unexpanded entries
        if (unexpanded & (before < 2u * width)) {
            if (before < width) {
                if (parents != nullptr) parents[before] = key_id(k);
                k |= 1ull;
            } else {
                next[before - width] = k;
            }
        }
        open_dst[r] = (uint16_t)(before > width ? before - width : 0u);
        dst[r] = k;
    }
};

// of the wave's mask the 16 bits of the lane's row, counted
__device__ __forceinline__ uint32_t count_row(uint64_t mask, uint32_t row) { return (uint32_t)__popc((uint32_t)(mask >> (16u * row)) & 0xFFFFu); }

// candidates ordered before `key`, 16 lanes a key, 32 candidates at a time (there is room for 64 keys past the list's end)
__device__ __forceinline__ uint32_t candidates_before(const Lds& l, uint64_t key, uint32_t nc, uint32_t row, uint32_t col) {
    uint32_t n = 0, s = 0;
    do {
        const uint64_t k0 = l.cand[s + col], k1 = l.cand[s + 16u + col];
        const uint64_t m0 = __ballot(k0 < key) & __ballot(s + col < nc), m1 = __ballot(k1 < key) & __ballot(s + 16u + col < nc);
        n += count_row(m0, row) + count_row(m1, row);
        s += 32;
    } while (s < nc);
    return n;
}

// Parents: 16 lanes a key, the unexpanded entries first (`ahead`: `width` of them in queue order, all-ones where there are
// fewer), then the candidates.  The merge drops as many entries from the end as there are candidates; a parent that
// is not clear of those (key not below `tail`) may be one of them: then M_TAIL says so, and the merge has to be made first.
struct Pick {
    uint64_t key, c0, c1, a0;
};
// what the first pass reads, whatever the number of candidates
__device__ __forceinline__ Pick pick_reads(const Lds& l, const uint64_t* ahead, uint32_t width, uint32_t x, uint32_t col) {
    return Pick{*(x < width ? ahead + x : l.cand + (x - width)), l.cand[col], l.cand[16u + col], ahead[col]};
}
template <int TB>
__device__ __forceinline__ void pick_parents(const Lds& l, Pick p, const uint64_t* ahead, uint32_t width, const uint64_t* queue, uint32_t itopk,
                                             uint32_t nc, int tid) {
    const uint32_t lane = (uint32_t)tid & 63u, row = lane >> 4, col = lane & 15u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    if (wave * 4u >= width + nc) return;
    uint64_t tail = queue[itopk - max(nc, 1u)] & ~1ull;
    if (nc == 0) tail = kInvalidKey;
    for (uint32_t x0 = wave * 4u;;) {
        const uint32_t x = x0 + row;
        uint32_t rank = count_row(__ballot(p.c0 < p.key) & __ballot(col < nc), row) + count_row(__ballot(p.c1 < p.key) & __ballot(16u + col < nc), row) +
                        count_row(__ballot(p.a0 < p.key) & __ballot(col < width), row);
        for (uint32_t s = 32; s < nc; s += 16) rank += count_row(__ballot(l.cand[s + col] < p.key) & __ballot(s + col < nc), row);
        for (uint32_t s = 16; s < width; s += 16) rank += count_row(__ballot(ahead[s + col] < p.key) & __ballot(s + col < width), row);
        if ((col == 0) & (x < width + nc) & (rank < width) & (p.key != kInvalidKey)) {
            l.parents[rank] = key_id(p.key);
            if (p.key >= tail) l.misc[M_TAIL] = 1;
        }
        x0 += TB / 16u;
        if (x0 >= width + nc) break;
        p = pick_reads(l, ahead, width, x0 + row, col);
    }
}

// A candidate's place, 16 lanes each: a look at every S-th queue entry and one at the S entries between two of those give
// the place in the queue.  `first`, `step4`: the keys that the wave takes.  MARK: note the place in the map.
template <bool MARK>
__device__ __forceinline__ void place_candidates(const Lds& l, const Merge& m, uint32_t itopk, uint32_t nc, uint32_t first, uint32_t stride,
                                                 uint32_t lane) {
    const uint32_t row = lane >> 4, col = lane & 15u;
    const uint32_t step = l.padded >> 4;  // S: 4, 8, 16 or 64
    for (uint32_t x0 = first; x0 < nc; x0 += stride) {
        const uint32_t x = x0 + row;
        const uint64_t c = l.cand[x];
        const uint64_t pivot = m.src[(col + 1u) * step - 1u] & ~1ull;  // an empty place stays above every candidate
        const uint32_t ahead = candidates_before(l, c, nc, row, col);
        const uint32_t lo = count_row(__ballot(pivot <= c), row) * step;
        uint32_t r = lo;
        for (uint32_t o = 0; o < step; o += 16) {  // past the block the entries are larger than c anyway
            const uint64_t k = m.src[min(lo + o + col, l.padded - 1u)] & ~1ull;
            r += count_row(__ballot(k <= c) & __ballot(o + col < step), row);
        }
        const uint32_t f = r + ahead;
        if ((col == 0) & (x < nc) & (f < itopk)) {  // a listed candidate beats the last entry, so r < itopk
            if (MARK) atomicOr(reinterpret_cast<uint32_t*>(l.marked) + (f >> 5), 1u << (f & 31u));
            m.place(c, f, m.open_src[r] + ahead, true);
        }
    }
}

// The queue's side of the merge where the candidates' places are marked: a place of the merged queue per thread; unless
// a candidate has it, it is the entry that has as many places before its own as there are unmarked ones before this.
template <int TB>
__device__ __forceinline__ void move_entries(const Lds& l, const Merge& m, uint32_t itopk, int tid) {
    for (uint32_t f = tid; f < itopk; f += TB) {
        const uint32_t block = (uint32_t)__builtin_amdgcn_readfirstlane((int)(f >> 6));
        const uint64_t mine = l.marked[block];
        uint32_t before = 0;
        for (uint32_t s = 0; s < block; ++s) before += (uint32_t)__popcll(l.marked[s]);
        const uint64_t bit = 1ull << (f & 63u);
        before += (uint32_t)__popcll(mine & (bit - 1ull));
        if (mine & bit) continue;
        const uint64_t k = m.src[f - before];
        m.place(k, f, m.open_src[f - before] + before, ((uint32_t)k & 1u) == 0u);  // an empty place holds the all-ones key
    }
}

// ... and on its own: 64 entries a wave, each counts the candidates ordered before it (all lanes read the list at one
// address).
__device__ __forceinline__ void shift_entries(const Lds& l, const Merge& m, uint32_t itopk, uint32_t nc, uint32_t block, uint32_t lane) {
    const uint32_t e = block * 64u + lane;
    const uint64_t k = m.src[e], kn = k & ~1ull;
    const uint32_t op = m.open_src[e];
    uint32_t cnt = 0;
    for (uint32_t c = 0; c < nc; c += 8) {
        uint64_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = l.cand[c + u];
#pragma unroll
        for (int u = 0; u < 8; ++u) cnt += (c + u < nc) & (v[u] < kn) ? 1u : 0u;
    }
    if (e + cnt < itopk) m.place(k, e + cnt, op + cnt, ((uint32_t)k & 1u) == 0u);
}

template <int TB, int CPL, int METRIC, int FILTER, bool FILL>
__global__ void __launch_bounds__(TB) search_small_kernel(const SearchArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr uint32_t W = TB / 64;
    const Lds l = carve(smem, a);
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t q = blockIdx.x;
    const bool filter_first = (a.flags & GRAB_FLAG_FILTER_FIRST) && FILTER != kFilterNone;
    const uint32_t itopk = a.itopk, width = a.search_width;
    const uint32_t table_size = 1u << a.table_bitlen;

    auto clear_table = [&]() {
        uint4* t4 = reinterpret_cast<uint4*>(l.table);  // 16 slots at least
        for (uint32_t i = tid; i < table_size / 4; i += TB) t4[i] = make_uint4(kInvalidId, kInvalidId, kInvalidId, kInvalidId);
    };
    // ---- set-up: query, empty queue, empty visited set (search.cu:217-227) ----
    {
        const float* gq = a.queries + (size_t)q * a.dim;
        for (uint32_t i = tid; i < a.dim; i += TB) l.query[i] = gq[i];
        for (uint32_t i = tid; i < 2u * l.padded; i += TB) {
            l.top[i] = kInvalidKey;
            l.open[i] = 0;
        }
        for (uint32_t i = tid; i < width; i += TB) {
            l.parents[i] = kInvalidId;
            l.ahead[i] = l.ahead[width + i] = kInvalidKey;
        }
        if (tid < 16) l.marked[tid] = 0;
        clear_table();
        if (tid < M_COUNT) l.misc[tid] = 0;
    }
    __syncthreads();

    float4 qreg[CPL ? CPL : 1];
    if (CPL > 0) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) qreg[c] = reinterpret_cast<const float4*>(l.query)[c * 8 + (lane & 7)];
    }

    FilterState<FILTER> flt{0, 0, 0};
    if (FILTER == kFilterRange || FILTER == kFilterIdRange || FILTER == kFilterRank) {
        flt.start = a.per_query_window ? a.win_start_arr[q] : a.win_start;
        flt.end = a.per_query_window ? a.win_end_arr[q] : a.win_end;
    } else if (FILTER == kFilterMask) {
        flt.mask = a.masks[q];
    }

    uint32_t my_f = 0, my_full = 0, my_par = 0;           // per-thread counts, reduced at the end
    uint32_t c_iters = 0, c_seed = 0, c_child = 0;        // uniform

    // The visited set takes 2^hash_bitlen ids and then no more (the table may have more slots than that, which only keeps
    // the probe sequences short).  Where so many can come at all (FILL) they are counted.  Where every id that enters
    // survives - no filter, or the filter comes first - the survivors' count does it, and of a phase's survivors as many
    // are taken as the set had room for; else a counter does, and an id waits for its place in the count.  An instance of
    // its own (SearchArgs::set_may_fill) because the others save the counting: 100 queries inside a window, itopk 128,
    // width 4, 100k x 128: 117 us without it, 126 with the counter that does not refuse ids one by one.
    const bool counting = FILL && FILTER != kFilterNone && !filter_first;
    uint32_t used = 0;  // uniform: FILL and not counting
    auto taken = [&](uint32_t came) {
        if (!FILL || counting) return came;
        const uint32_t left = (1u << a.hash_bitlen) - used;
        if (came > left) {
            if (tid == 0) my_full += came - left;
            came = left;
        }
        used += came;
        return came;
    };
    auto enter = [&](bool active, uint32_t id, bool counted) {
        const bool full = FILL && (counted ? __atomic_load_n(&l.misc[M_USED], __ATOMIC_RELAXED) : used) >> a.hash_bitlen;
        int r = 0;
        if (active) r = hash_insert<false>(l.table, a.table_bitlen, id, full);
        if (FILL && counted && r == 1 && lds_append(&l.misc[M_USED]) >> a.hash_bitlen) r = -1;
        if (FILL && r < 0) my_full++;
        return r == 1;
    };
    // one id per thread: visited set, filter, survivor list
    auto visit = [&](bool keep, uint32_t id) {
        if (filter_first && keep) {
            if (FILTER != kFilterIdRange) my_f++;
            keep = filter_pass<FILTER>(a, flt, id);
        }
        keep = enter(keep, id, counting);
        if (FILTER != kFilterNone && !filter_first && keep) {
            if (FILTER != kFilterIdRange) my_f++;
            keep = filter_pass<FILTER>(a, flt, id);
        }
        if (keep) l.surv[lds_append(&l.misc[M_NSURV])] = id;
    };
    auto score = [&](uint32_t ns, uint64_t worst, uint32_t* ncand) {
        for (uint32_t s0 = wave * 8u; s0 < ns; s0 += 2u * W * 8u) {
            if (s0 + W * 8u < ns) score_round<CPL, METRIC, true>(a, l, qreg, ns, s0, W * 8u, worst, ncand, lane);
            else score_round<CPL, METRIC, false>(a, l, qreg, ns, s0, 0, worst, ncand, lane);
        }
    };

    // ---- seeds (compute_distance.cuh:144-202, :204-269) ----
    for (uint32_t base = wave * 64u; base < a.n_seeds; base += TB) {
        const uint32_t i = base + lane;
        uint32_t id = kInvalidId;
        if (i < a.n_seeds) {
            if (a.seeds != nullptr && i < a.n_provided) id = a.seeds[(size_t)q * a.n_provided + i];
            if ((uint64_t)id >= a.n) id = (uint32_t)((a.rand_xor_mask * (uint64_t)(i + 1)) % a.n);
        }
        visit(i < a.n_seeds, id);
    }
    __syncthreads();
    c_seed = taken((uint32_t)__builtin_amdgcn_readfirstlane((int)l.misc[M_NSURV]));
    score(c_seed, kInvalidKey, &l.misc[M_NCAND]);
    __syncthreads();

    uint32_t cur = 0;     // which half of `top` holds the queue: 0 or `padded`
    uint32_t turn = 0;    // which counter and list are in use
    bool pending = true;  // candidates that are not in the queue yet
    // Candidates that are merged beside the expansion: waves that have no neighbours to read, up to 48 candidates (a wave
    // of queue entries takes about five instructions for each).
    const uint32_t readers = (width * a.degree + 63u) >> 6, blocks = (itopk + 63u) >> 6;
    const bool beside = readers + blocks + 2u <= W;
    auto merge_of = [&](uint32_t w, uint32_t* parents) {
        const uint32_t to = l.padded - cur;
        return Merge{l.top + cur, l.top + to, l.open + cur, l.open + to, w, parents, l.ahead + (turn ^ 1u) * width};
    };
    auto merge_all = [&](uint32_t w, uint32_t nc) {
        const Merge m = merge_of(w, l.parents);
        place_candidates<true>(l, m, itopk, nc, wave * 4u, W * 4u, (uint32_t)lane);
        __syncthreads();
        move_entries<TB>(l, m, itopk, tid);
        __syncthreads();
        cur = l.padded - cur;
    };
    for (uint32_t iter = 0; iter < a.max_iterations; ++iter) {
        const uint64_t* ahead = l.ahead + turn * width;
        const Pick first = pick_reads(l, ahead, width, wave * 4u + ((uint32_t)lane >> 4), (uint32_t)lane & 15u);
        const uint32_t open0 = (uint32_t)ahead[0], listed = l.misc[M_NCAND + turn];
        const uint32_t nc = (uint32_t)__builtin_amdgcn_readfirstlane((int)listed);
        const bool rebuild = iter > 0 && (iter % 30u == 0);
        bool split = beside && nc <= 48u && nc <= itopk && !rebuild;
        if (nc == 0 && __builtin_amdgcn_readfirstlane((int)open0) == -1) {  // nothing is left to expand
            pending = false;
            break;
        }
        if (tid == TB - 1) l.misc[M_NSURV] = 0;  // read by the scoring before this, added to after a barrier
        if (split) {
            pick_parents<TB>(l, first, ahead, width, l.top + cur, itopk, nc, tid);
            __syncthreads();
            split = l.misc[M_TAIL] == 0;
            if (!split) {
                for (uint32_t i = tid; i < width; i += TB) l.parents[i] = kInvalidId;
                __syncthreads();
            }
        }
        if (!split) {
            merge_all(width, nc);
            if (l.parents[0] == kInvalidId) {  // what was unexpanded fell off the end
                pending = false;
                break;
            }
        }
        if (rebuild) {  // the visited set is rebuilt from the queue (search.cu:265-283, hashmap.cuh:103-117)
            clear_table();
            if (tid == 0) l.misc[M_USED] = 0;
            used = 0;
            __syncthreads();
            for (uint32_t base = 0; base < itopk; base += TB) {
                const uint32_t i = base + tid;
                const uint64_t k = i < itopk ? l.top[cur + i] : kInvalidKey;
                (void)enter(k != kInvalidKey, key_id(k), FILL);
            }
            __syncthreads();
            if (FILL) used = min((uint32_t)__builtin_amdgcn_readfirstlane((int)l.misc[M_USED]), 1u << a.hash_bitlen);
        }
        c_iters++;

        // ---- expansion: ids, visited set, filter (compute_distance.cuh:274-380 etc.) ----
        for (uint32_t base = wave * 64u; base < width * a.degree; base += TB) {
            const uint32_t t = base + lane;
            uint32_t p, off;
            if (a.degree_shift < 32u) {
                p = t >> a.degree_shift;
                off = t & (a.degree - 1u);
            } else {
                p = t / a.degree;
                off = t - p * a.degree;
            }
            const uint32_t parent = p < width ? l.parents[p] : kInvalidId;
            uint32_t id = kInvalidId;
            if (parent != kInvalidId && off < a.active_degree) id = a.graph[(size_t)parent * a.degree + off];  // compute_distance.cuh:428-436
            visit((uint64_t)id < a.n, id);
        }
        if (split) {
            if (wave >= readers) {
                const Merge m = merge_of(width, nullptr);
                const uint32_t w = wave - readers;
                if (w < blocks) shift_entries(l, m, itopk, nc, w, (uint32_t)lane);
                else place_candidates<false>(l, m, itopk, nc, (w - blocks) * 4u, (W - readers - blocks) * 4u, (uint32_t)lane);
            }
            cur = l.padded - cur;
        }
        __syncthreads();
        const uint32_t ns = taken((uint32_t)__builtin_amdgcn_readfirstlane((int)l.misc[M_NSURV]));
        c_child += ns;
        // what the phases before have read starts again
        if (tid >= TB - 16) l.marked[TB - 1 - tid] = 0;
        if (tid == 0) l.misc[M_NCAND + turn] = l.misc[M_TAIL] = 0;
        for (uint32_t i = TB - 1 - tid; i < width; i += TB) {
            my_par += l.parents[i] != kInvalidId ? 1u : 0u;
            l.parents[i] = kInvalidId;
            l.ahead[turn * width + i] = kInvalidKey;
        }
        turn ^= 1u;
        score(ns, l.top[cur + itopk - 1] & ~1ull, &l.misc[M_NCAND + turn]);
        __syncthreads();
    }
    if (pending) merge_all(0, (uint32_t)__builtin_amdgcn_readfirstlane((int)l.misc[M_NCAND + turn]));

    // ---- results (search.cu:348-355; ids widened here instead of a second kernel) ----
    for (uint32_t r = tid; r < a.k; r += TB) {
        const uint64_t k = l.top[cur + r];
        int64_t id = -1;
        float d = kDistMax;
        if (k != kInvalidKey) {
            id = (int64_t)key_id(k);
            d = key_dist(k);
        }
        a.out_ids[(size_t)q * a.k + r] = id;
        a.out_dists[(size_t)q * a.k + r] = d;
    }

    if (a.counters != nullptr) {
        if (my_par) atomicAdd(&l.misc[M_PAR], my_par);
        if (my_f) atomicAdd(&l.misc[M_F], my_f);
        if (my_full) atomicAdd(&l.misc[M_FULL], my_full);
        __syncthreads();
        if (tid == 0) {
            grab_counters* c = a.counters + q;
            c->iterations = c_iters;
            c->seed_dists = c_seed;
            c->parents = l.misc[M_PAR];
            c->filter_reads = l.misc[M_F];
            c->child_dists = c_child;
            c->hash_full = l.misc[M_FULL];
        }
    }
}

template <int CPL, int METRIC, int FILTER>
int launch(const SearchArgs& a, size_t lds_bytes, hipStream_t stream) {
    auto kern = a.threads == 1024 ? (a.set_may_fill ? search_small_kernel<1024, CPL, METRIC, FILTER, true> : search_small_kernel<1024, CPL, METRIC, FILTER, false>)
                                  : (a.set_may_fill ? search_small_kernel<512, CPL, METRIC, FILTER, true> : search_small_kernel<512, CPL, METRIC, FILTER, false>);
    if (lds_bytes > 64 * 1024)
        GRAB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
    hipLaunchKernelGGL(kern, dim3(a.nq), dim3(a.threads), lds_bytes, stream, a);
    GRAB_HIP(hipGetLastError());
    return GRAB_OK;
}

template <int CPL>
int dispatch_mf(const SearchArgs& a, int metric, int filter, size_t lds, hipStream_t s) {
#define GRAB_CASE(M, F) \
    if (metric == M && filter == F) return launch<CPL, M, F>(a, lds, s);
    GRAB_CASE(kMetricL2, kFilterNone)
    GRAB_CASE(kMetricL2, kFilterRange)
    GRAB_CASE(kMetricL2, kFilterMask)
    GRAB_CASE(kMetricL2, kFilterIdRange)
    GRAB_CASE(kMetricL2, kFilterRank)
    GRAB_CASE(kMetricIP, kFilterNone)
    GRAB_CASE(kMetricIP, kFilterRange)
    GRAB_CASE(kMetricIP, kFilterMask)
    GRAB_CASE(kMetricIP, kFilterIdRange)
    GRAB_CASE(kMetricIP, kFilterRank)
#undef GRAB_CASE
    set_error("unsupported metric %d / filter %d", metric, filter);
    return GRAB_ERR_INVALID;
}

}  // namespace

int launch_search_small(const SearchArgs& a, int metric, int filter, size_t lds_bytes, hipStream_t stream) {
    if (a.dim == 128) return dispatch_mf<4>(a, metric, filter, lds_bytes, stream);
    return dispatch_mf<0>(a, metric, filter, lds_bytes, stream);
}

}  // namespace grab
