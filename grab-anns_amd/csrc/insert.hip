// Incremental insert into the global graph.  Restates cagra::insert
// (src/index/cagra.cu:938-1015) with find_near_nodes and update_topology_gpu_v1
// (src/index/insert.cu:140-440): search the old graph with the new rows as queries, re-score
// and sort the results, write the new rows, then let every old node that was found take the
// new node into a pseudo-random slot of its own row.
#include <algorithm>

#include "device_sort.hpp"
#include "insert_internal.hpp"
#include "search_internal.hpp"

namespace grab {
using namespace dev;
namespace {

// insert_refine_kernel_warp + insert_sort_kernel (insert.cu:24-72, :80-133), one workgroup per new
// row: its four waves score the result list 32 entries at a time (8 lanes per entry), the first wave
// sorts.  Ids outside [0, n_existing) score kDistMax; the sort carries ids as uint32 and widens
// them again (insert.cu:106,129).  With `striped` the output slot p = lane32 + e*32 receives
// the element of sorted rank lane32*per_lane + e, which is what the reference's striped load
// into a blocked 32-lane network produces (insert.cu:104 against bitonic.cuh:74).
//
// fill_new_nodes_kernel (insert.cu:225-257) and generate_update_requests_kernel (:263-290) follow in the same wave: the
// new graph row, and the row's update requests.  A request is the 64-bit key target<<32 | request index: sorting the keys
// groups requests by target and keeps their original order inside a group, which is what a stable sort_by_key on the
// 32-bit target gives (:422-424).  The wave leaves its own requests sorted, which turns the sort of all of them into
// searches in sorted runs (merge_runs_kernel): a second register sort here, 11.8 us, for a kernel of 8.9 and one of 4.7.
template <int METRIC, int NPL>
__global__ void __launch_bounds__(256) insert_refine_sort_kernel(const float* __restrict__ data, const float* __restrict__ new_data,
                                                                 uint32_t dim, uint32_t n_existing, uint32_t n_new,
                                                                 uint32_t search_k, const int64_t* __restrict__ ids, int striped,
                                                                 uint32_t per_lane32, uint32_t* __restrict__ graph, uint32_t degree,
                                                                 uint64_t* __restrict__ requests) {
    __shared__ uint64_t mykeys[64 * NPL];
    const int lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x;
    const int64_t* myids = ids + (size_t)row * search_k;
    const float* q = new_data + (size_t)row * dim;
    const int grp = threadIdx.x >> 3, j = threadIdx.x & 7;
    for (uint32_t g = threadIdx.x; g < 64u * NPL; g += 256) mykeys[g] = kInvalidKey;
    __syncthreads();
    for (uint32_t c0 = 0; c0 < search_k; c0 += 32) {
        const uint32_t c = c0 + grp;
        if (c < search_k) {  // uniform per group of 8 lanes
            const int64_t id = myids[c];
            float d = kDistMax;
            if (id >= 0 && id < (int64_t)n_existing) d = group8_distance<METRIC>(q, data + (size_t)id * dim, dim, j);
            if (j == 0) mykeys[c] = make_sel_key(d, (uint32_t)id);
        }
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    uint64_t k[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) k[i] = mykeys[lane * NPL + i];
    wave_bitonic_sort<NPL>(k);
#pragma unroll
    for (int i = 0; i < NPL; ++i) mykeys[lane * NPL + i] = k[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
        const uint32_t p = lane + 64u * i;
        uint32_t src = p;
        if (striped) src = (p & 31u) * per_lane32 + (p >> 5);
        // ranks past search_k are the (FLT_MAX, 0xFFFFFFFF) padding of the reference's network
        const uint32_t id = p < search_k && src < search_k ? (uint32_t)(mykeys[src] & 0xFFFFFFFFull) : kInvalidId;
        const bool old_node = id < n_existing;
        if (p < min(degree, search_k)) graph[(size_t)(n_existing + row) * degree + p] = old_node ? id : kInvalidId;
        k[i] = old_node ? (((uint64_t)id << 32) | (row * search_k + p)) : kInvalidKey;
    }
    wave_bitonic_sort<NPL>(k);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
        const uint32_t g = lane * NPL + i;
        if (g < search_k) requests[(size_t)row * search_k + g] = k[i];
    }
}

// All requests in ascending order, from the rows' sorted runs: a key's place is the number of keys ordered before it
// (smaller, or equal - invalid ones only - in an earlier run), found by sixteen lanes that search every sixteenth run of a
// copy in LDS, four runs at a time.  Bound by the copy and by a chain of eight LDS reads, where counting over all keys
// reads each of them for each: 8192 keys, 19 -> 6.9 us.  Runs start an odd number of keys apart, so that lanes at the same place of different runs use different banks.
constexpr uint32_t kRunLanes = 16, kRunThreads = 1024;
constexpr size_t kRunLdsMax = 144 * 1024;
__global__ void __launch_bounds__(kRunThreads) merge_runs_kernel(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint32_t runs,
                                                                 uint32_t len) {
    extern __shared__ uint64_t sk[];
    const uint32_t n = runs * len, pitch = len | 1u;
    for (uint32_t i = threadIdx.x; i < n; i += kRunThreads) {
        const uint32_t r = i / len;
        sk[r * pitch + (i - r * len)] = in[i];
    }
    __syncthreads();
    const uint32_t i = blockIdx.x * (kRunThreads / kRunLanes) + threadIdx.x / kRunLanes, s = threadIdx.x % kRunLanes;
    const uint32_t my_run = min(i, n - 1u) / len, my_pos = min(i, n - 1u) - my_run * len;
    const uint64_t mine = sk[my_run * pitch + my_pos];
    const uint32_t top = 1u << (31 - __clz((int)len));
    uint32_t cnt = 0;
    for (uint32_t r0 = s; r0 < runs; r0 += 4 * kRunLanes) {
        uint32_t lo[4] = {0, 0, 0, 0};
        for (uint32_t step = top; step > 0; step >>= 1) {
            uint64_t v[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) v[u] = sk[min(r0 + u * kRunLanes, runs - 1u) * pitch + min(lo[u] + step, len) - 1u];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const bool before = v[u] < mine || (v[u] == mine && r0 + u * kRunLanes < my_run);
                if (before && lo[u] + step <= len) lo[u] += step;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t r = r0 + u * kRunLanes;
            if (r < runs) cnt += r == my_run ? my_pos : lo[u];
        }
    }
#pragma unroll
    for (int m = 1; m < (int)kRunLanes; m <<= 1) cnt += __shfl_xor(cnt, m, 64);
    if (s == 0 && i < n) out[cnt] = mine;
}

__global__ void __launch_bounds__(256) fill_invalid_kernel(uint64_t* __restrict__ keys, uint32_t count) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t < count) keys[t] = kInvalidKey;
}

// new rows wider than the result list keep 0xFFFFFFFF in the slots past search_k (insert.cu:245)
__global__ void __launch_bounds__(256) fill_tail_kernel(uint32_t* __restrict__ graph, uint32_t n_existing, uint32_t n_new,
                                                        uint32_t degree, uint32_t search_k) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    const uint32_t width = degree - search_k;
    if (t >= n_new * width) return;
    const uint32_t i = t / width, kk = search_k + (t - i * width);
    graph[(size_t)(n_existing + i) * degree + kk] = kInvalidId;
}

// apply_topology_updates_kernel (insert.cu:296-368): the first request of each target walks
// the target's requests in order; a new id that is not yet in the row overwrites a slot
// drawn from a 64-bit LCG seeded with target*0x9e3779b97f4a7c15 + position of the leader:
// one time in ten a slot of the first half, otherwise one of the second half.
// Sixteen lanes per request, those of a target's first one go on.  Latency-bound: the target's row is read once, in one
// piece, into registers (NE slots a lane) and kept up to date there, and sixteen of the target's requests come with one
// read, so a chain of requests waits for no memory.  8192 requests, degree 64: 18 -> 7.2 us against a thread per request.
template <int NE>
__global__ void __launch_bounds__(256) apply_updates_kernel(uint32_t* __restrict__ graph, const uint64_t* __restrict__ sorted,
                                                            uint32_t total, uint32_t degree, uint32_t n_existing,
                                                            uint32_t search_k) {
    const uint32_t first = blockIdx.x * 16 + threadIdx.x / 16, l = threadIdx.x & 15u;
    const int lane = threadIdx.x & 63, group = lane & 48;
    if (first >= total) return;  // uniform over the sixteen lanes, as every branch below
    const uint64_t key = sorted[first], before = first != 0 ? sorted[first - 1] : kInvalidKey;
    uint64_t mine = first + l < total ? sorted[first + l] : kInvalidKey;
    if (key == kInvalidKey) return;
    const uint32_t target = (uint32_t)(key >> 32);
    if (first != 0 && (uint32_t)(before >> 32) == target) return;  // not the target's first request
    uint32_t* nb = graph + (size_t)target * degree;
    uint32_t e[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) e[i] = l + 16u * i < degree ? nb[l + 16u * i] : kInvalidId;
    const uint32_t num_protected = degree / 2, num_unprotected = degree - num_protected;
    uint64_t rng = (uint64_t)target * 0x9e3779b97f4a7c15ull + (uint64_t)first;
    for (uint32_t at = first;;) {
        const bool same = mine != kInvalidKey && (uint32_t)(mine >> 32) == target;
        const uint32_t marks = (uint32_t)(__ballot(same) >> group) & 0xFFFFu;
        const uint32_t count = (uint32_t)__builtin_ctz(~marks);  // the target's requests follow each other
        for (uint32_t c = 0; c < count; ++c) {
            const uint32_t nid = n_existing + (uint32_t)__shfl((int)(uint32_t)mine, group + (int)c, 64) / search_k;
            bool exists = false;
#pragma unroll
            for (int i = 0; i < NE; ++i) exists |= e[i] == nid;
            if (((__ballot(exists) >> group) & 0xFFFFull) != 0) continue;
            rng = rng * 6364136223846793005ull + 1;
            const uint32_t r1 = (uint32_t)(rng >> 32);
            const bool upd_protected = (r1 % 10u == 0) && num_protected != 0;  // a row of one slot has no first half
            rng = rng * 6364136223846793005ull + 1;
            const uint32_t r2 = (uint32_t)(rng >> 32);
            const uint32_t slot = upd_protected ? (r2 % num_protected) : num_protected + (r2 % num_unprotected);
            if (l == (slot & 15u)) {
                nb[slot] = nid;
#pragma unroll
                for (int i = 0; i < NE; ++i)
                    if (slot / 16u == (uint32_t)i) e[i] = nid;
            }
        }
        at += 16;
        if (count < 16 || at >= total) break;
        mine = at + l < total ? sorted[at + l] : kInvalidKey;
    }
}

template <int METRIC>
int launch_refine_sort(const float* data, const float* new_data, uint32_t dim, uint32_t n_existing, uint32_t n_new,
                       uint32_t search_k, const int64_t* ids, int striped, uint32_t* graph, uint32_t degree, uint64_t* requests, hipStream_t st) {
    const uint32_t grid = n_new;
    const uint32_t per_lane32 = search_k <= 64 ? 2 : search_k <= 128 ? 4 : search_k <= 256 ? 8 : 16;  // insert.cu:204-213
#define GRAB_RS(NPL) \
    hipLaunchKernelGGL((insert_refine_sort_kernel<METRIC, NPL>), dim3(grid), dim3(256), 0, st, data, new_data, dim, n_existing, n_new, search_k, ids, striped, per_lane32, graph, degree, requests)
    if (search_k <= 64) GRAB_RS(1);
    else if (search_k <= 128) GRAB_RS(2);
    else if (search_k <= 256) GRAB_RS(4);
    else if (search_k <= 512) GRAB_RS(8);
    else GRAB_RS(16);
#undef GRAB_RS
    GRAB_HIP(hipGetLastError());
    return GRAB_OK;
}

}  // namespace

size_t insert_workspace_bytes(size_t num_new, uint32_t degree) {
    const size_t search_k = (size_t)degree * 2;
    const size_t total = num_new * search_k;
    const size_t padded = grab_next_power_of_2((uint32_t)std::max<size_t>(total, 2));
    return total * sizeof(int64_t) + total * sizeof(float) + 2 * padded * sizeof(uint64_t) + 256;
}

int insert_impl(const float* d_dataset, uint32_t dim, size_t num_existing, size_t num_new, const float* d_new_data,
                uint32_t* d_graph, uint32_t degree, grab_search_params params, int metric, uint64_t* rng_state,
                uint32_t flags, int striped_sort, void* workspace, hipStream_t st) {
    if (num_new == 0) return GRAB_OK;
    GRAB_REQUIRE(d_dataset && d_new_data && d_graph && rng_state && workspace, "null pointer");
    GRAB_REQUIRE(num_existing > 0, "insert needs an existing graph");
    GRAB_REQUIRE(degree >= 1 && degree <= GRAB_MAX_DEGREE, "graph_degree %u out of range", degree);
    const uint32_t search_k = degree * 2;  // cagra.cu:951
    GRAB_REQUIRE(search_k <= 1024, "graph_degree above 512 is not supported");
    GRAB_REQUIRE(num_new * (size_t)search_k < (1ull << 31), "too many new rows in one call");
    GRAB_REQUIRE(num_existing + num_new < (1ull << 31), "index too large");
    const uint32_t n_existing = (uint32_t)num_existing, n_new = (uint32_t)num_new;
    const uint32_t total = n_new * search_k;
    const uint32_t padded = grab_next_power_of_2(std::max(total, 2u));

    char* ws = static_cast<char*>(workspace);
    int64_t* ids = reinterpret_cast<int64_t*>(ws);
    ws += (size_t)total * sizeof(int64_t);
    uint64_t* requests = reinterpret_cast<uint64_t*>(ws);
    ws += (size_t)padded * sizeof(uint64_t);
    uint64_t* sorted = reinterpret_cast<uint64_t*>(ws);
    ws += (size_t)padded * sizeof(uint64_t);
    float* dists = reinterpret_cast<float*>(ws);

    // find_near_nodes (insert.cu:140-219): one search per 64 new rows, each with its own mask
    for (size_t off = 0; off < num_new; off += 64) {
        const size_t cur = std::min<size_t>(64, num_new - off);
        const uint64_t mask = splitmix64(rng_state) & 0xFFFFFFFFull;
        grab_search_desc d;
        fill_search_desc(&d, GRAB_WRAP_SEARCH, d_dataset, num_existing, dim, d_graph, degree, degree,
                         d_new_data + off * dim, cur, search_k, params, metric, nullptr, 0, mask, flags,
                         ids + off * search_k, dists + off * search_k, st);
        GRAB_TRY(search_ex_impl(&d, false));
    }
    if (metric == kMetricIP)
        GRAB_TRY(launch_refine_sort<kMetricIP>(d_dataset, d_new_data, dim, n_existing, n_new, search_k, ids, striped_sort, d_graph, degree, requests, st));
    else
        GRAB_TRY(launch_refine_sort<kMetricL2>(d_dataset, d_new_data, dim, n_existing, n_new, search_k, ids, striped_sort, d_graph, degree, requests, st));

    if (degree > search_k)
        hipLaunchKernelGGL(fill_tail_kernel, dim3((n_new * (degree - search_k) + 255) / 256), dim3(256), 0, st, d_graph,
                           n_existing, n_new, degree, search_k);
    const size_t run_lds = (size_t)n_new * (search_k | 1u) * sizeof(uint64_t);
    if (run_lds <= kRunLdsMax && n_new <= 1024) {  // more runs: a key would search more of them than counting costs
        if (run_lds > 64 * 1024)
            GRAB_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(merge_runs_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)run_lds));
        const uint32_t per = kRunThreads / kRunLanes;
        hipLaunchKernelGGL(merge_runs_kernel, dim3((total + per - 1) / per), dim3(kRunThreads), run_lds, st, requests, sorted, n_new, search_k);
    } else {
        if (padded > total)
            hipLaunchKernelGGL(fill_invalid_kernel, dim3((padded - total + 255) / 256), dim3(256), 0, st, requests + total, padded - total);
        GRAB_TRY(rank_sort_u64_async(requests, sorted, padded, st));
    }
    auto apply = degree <= 64 ? apply_updates_kernel<4> : degree <= 128 ? apply_updates_kernel<8> : degree <= 256 ? apply_updates_kernel<16> : apply_updates_kernel<32>;
    hipLaunchKernelGGL(apply, dim3((total + 15) / 16), dim3(256), 0, st, d_graph, sorted, total, degree, n_existing, search_k);
    GRAB_HIP(hipGetLastError());
    return GRAB_OK;
}

}  // namespace grab

using namespace grab;

extern "C" {

int grab_insert(const float* d_dataset, uint32_t dim, size_t num_existing, size_t num_new, const float* d_new_data,
                uint32_t* d_graph, uint32_t graph_degree, grab_search_params params, int metric, uint64_t* rng_state,
                uint32_t flags, int striped_sort, void* stream) {
    if (num_new == 0) return GRAB_OK;
    GRAB_REQUIRE(graph_degree >= 1 && graph_degree <= GRAB_MAX_DEGREE, "graph_degree %u out of range", graph_degree);
    DeviceScratch ws;
    GRAB_HIP(ws.alloc(insert_workspace_bytes(num_new, graph_degree)));
    hipStream_t st = static_cast<hipStream_t>(stream);
    GRAB_TRY(insert_impl(d_dataset, dim, num_existing, num_new, d_new_data, d_graph, graph_degree, params, metric, rng_state,
                         flags, striped_sort, ws.ptr, st));
    GRAB_HIP(hipStreamSynchronize(st));
    return GRAB_OK;
}

}  // extern "C"
