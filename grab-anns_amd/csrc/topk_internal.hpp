// What the translation units around the tile contraction share (topk_gemm.hip: the kernels, exact_topk; entry_layer.hip:
// the entry-point layer; scan.hip: the exact scans of buckets and id intervals): tile geometry, the argument blocks of
// the contraction and of the re-scoring, and launchers that pick the kernel instance.
#pragma once
#include <cstdint>
#include <vector>

#include "common.hpp"
#include "topk_gemm.hpp"

namespace grab {

constexpr int TM = 128, TN = 128, KC = 32, LDS_STRIDE = KC + 4;
constexpr int TSTRIDE = 68;               // row stride of the transposed 64x64 block: 16-byte aligned rows, conflict-free b128 reads
constexpr int CAP = 1024;                 // per-row candidate buffer (keys)
constexpr int COMPACT_AT = CAP - TN;      // a tile appends at most TN keys to a row
// layout of the work list of the dense-store mode (uint32 words)
constexpr int kSchedPer = 0, kSchedItems = 1, kSchedOff = 2, kSchedLo = kSchedOff + 129, kSchedHi = kSchedLo + 128,
              kSchedBase = kSchedHi + 128, kSchedWords = kSchedBase + 128;

struct TileArgs {
    const float* A;
    const float* B;
    const float* normA;
    const float* normB;
    const uint64_t* ts;
    const uint64_t* win_start_arr;
    const uint64_t* win_end_arr;
    const uint8_t* labels;
    const uint64_t* masks;
    const uint32_t* row_perm;  // optional: tile-grid row -> row of A (rows ordered by window)
    const uint32_t* row_lo;    // kFilterColRange: per row of A, admissible columns [lo,hi)
    const uint32_t* row_hi;
    float* dense;        // STORE mode: [M][dense_pitch] distances
    uint64_t dense_pitch;
    // STORE mode: a row tile is a matrix of its own, as wide as its sweep; they follow each other (sched has the column
    // tiles before each), dense_pitch is not used, and only columns that a row admits are written
    int dense_rel;
    const uint32_t* sched;  // STORE mode: work list made by bucket_order_kernel
    uint64_t* buf;       // [gridDim.x][TM][CAP]
    uint64_t* cand_out;  // [M][nsplit*kk]
    // kFilterSymmetric: what a tile above the diagonal yields for the rows behind its columns
    const float* col_bound;  // [N] a row takes a key from a column walk when its distance is <= this
    uint64_t* col_list;      // [N][col_cap] keys (distance, row of A), in arrival order
    uint32_t* col_count;     // [N] keys offered to a row (may exceed col_cap: the row is then redone the plain way)
    uint32_t col_cap;
    // optional, zero before the launch: work items are handed out through it in their order, to whichever workgroup is
    // free, instead of in equal shares (the two workgroups of a CU do not run at the same pace)
    uint32_t* work_counter;
    int cand_by_grid_row;    // cand_out is indexed by the tile-grid row instead of the row of A
    int range_by_grid_row;   // kFilterColRange: so are row_lo / row_hi (several tile-grid rows may stand for one row of A)
    uint64_t win_start, win_end;
    uint32_t M, N, dim, kk, nsplit, col_tiles, tiles_per_split, row_tiles;
    int per_query_window;
};

struct RefineArgs {
    const float* A;
    const float* B;
    const uint64_t* cand;  // [M][nc]
    uint32_t* out_u32;     // kNN mode: [M][k]
    int64_t* out_i64;      // top-k mode: [M][k]
    float* out_dist;
    uint32_t M, dim, nc, k;
    int drop_self;
    // certificate (optional): nc = nsplit lists of kk keys, each the kk smallest GEMM-form keys of its columns
    uint32_t kk;
    const float* normA;      // squared norm of every row of A
    const float* max_normB;  // one float: the largest squared norm among the rows of B
    // candidates that (may also) come from rows split into bf16 halves, centred or not: their norms, and the products' error
    const float* split_normA;      // null: none do
    const float* split_max_normB;
    float split_terms;             // products that one of its fp32 sums runs over (3 * dim)
    int sorted;                    // every row's candidates are one list in ascending order (the symmetric pass leaves them so)
    const float* outside_in; // optional, per row: a bound like `outside` below that the lists themselves no longer show (they were merged)
    uint32_t* doubt;         // rows whose result the candidates do not prove, doubt[0] = how many, then the rows; null = no check
    const uint32_t* rows;    // optional: only these rows (M of them)
    int cand_by_slot;        // ... whose candidates follow each other in cand, in that order
};

// selection inside the contraction (tile_topk_kernel<METRIC, FILTER, false, SPLIT>): a.cand_out receives kk keys per row and split
int launch_tile_any(const TileArgs& a, int metric, int filter, uint32_t grid, hipStream_t stream, bool split = false);
// distances of the swept columns to a.dense (tile_topk_kernel<METRIC, kFilterColRange, true, SPLIT>), work list in a.sched
int launch_tile_store(const TileArgs& a, int metric, uint32_t grid, hipStream_t stream, bool split = false);
int launch_refine_any(const RefineArgs& a, int metric, hipStream_t stream);
// squared norms of n rows; the largest of n non-negative floats (atomic max into *out, which the caller has zeroed);
// the mean of `count` evenly spaced rows; rows as bf16 halves per chunk of 32 dimensions (minus `mean` if given) and
// the squared norms of what was split
void launch_row_norms(const float* x, size_t n, uint32_t dim, float* out, hipStream_t stream);
void launch_max_float(const float* x, uint64_t n, uint32_t* out, hipStream_t stream);
void launch_spaced_mean(const float* data, uint64_t n, uint32_t count, uint32_t dim, float* mean, hipStream_t stream);
void launch_split_rows_chunked(const float* data, uint64_t n, uint32_t dim, const float* mean, uint16_t* out, float* norm,
                               hipStream_t stream);

// *flag: whether rows rounded to f16 tell their inner products apart less well than rows as bf16 halves (1 or 0).  scratch: dim + kOneWayRows floats
constexpr uint32_t kOneWayRows = 1024;
void launch_one_way(const float* data, uint64_t n, uint32_t dim, float* scratch, uint32_t* flag, hipStream_t stream);

// The candidates of a large kNN graph from f16 products: knn_half.hip.  Where it applies, a plan of the sizes, the lists, and
// the neighbours that these prove.
// words of `scal`: whether some row is not finite; whether one, not NaN, is too long to be packed; scans, inner product: launch_one_way's
constexpr uint32_t kScalBad = 11, kScalLong = 12, kScalOneWay = 13;
constexpr uint32_t kHalfListCap = 1024;  // keys of a row's list
constexpr uint32_t kHalfSample = 49152;  // sample rows that the bounds are taken from, at most
struct HalfKnn {
    uint32_t n = 0, dim = 0, places = 0, n_sample = 0, sample_places = 0, class_rank = 0, min_list = 0, id_bits = 0, ks = 0, frags = 0;
    bool ip = false;
    size_t workspace_bytes = 0, list_bytes = 0, at_blocks = 0, at_sample = 0, at_row_frags = 0, at_words = 0;
    // in the workspace: rows in blocks, by place (places are padded to whole tiles), and the sample's; per row its bound, the
    // squared norm of the centred row and what rounding moved it; per place the row, thresholds and the list's length;
    // scal: [0] the largest centred norm, [1] the largest rounding (both as float bits), [2 ..] work counters
    uint4* blocks = nullptr;
    uint4* sample_blocks = nullptr;
    uint4* row_frags = nullptr;
    float *best = nullptr, *centre = nullptr, *hn = nullptr, *cnorm = nullptr, *eps = nullptr, *bound = nullptr, *t_own = nullptr, *t_step = nullptr, *top = nullptr;
    uint32_t *perm = nullptr, *bins = nullptr, *count = nullptr, *scal = nullptr;
    uint32_t* list = nullptr;
};
bool half_knn_applies(uint64_t n, uint32_t dim, int metric);
int half_knn_plan(uint32_t n, uint32_t dim, uint32_t k, int metric, HalfKnn* h);
// queued on `st`: every row's columns within its bound to list[place][kHalfListCap]
int half_knn_lists_async(const float* data, HalfKnn* h, void* workspace, uint32_t* list, uint32_t num_cu, hipStream_t st);
// queued on `st`: out[row][k]; rows that their lists do not prove are listed in redo (a longer list may) or doubt[1..] (it
// cannot), their numbers in *redo_count and doubt[0], zero before.  norm, max_norm: of the rows as they are
int half_knn_finish_async(const float* data, const HalfKnn& h, uint32_t k, uint32_t redo_keep, const float* norm, const float* max_norm, uint32_t* out,
                          uint32_t* redo_count, uint32_t* redo, uint32_t* doubt, hipStream_t st);

// Queries against intervals of a row set, on f16 products: scan_half.hip.  The base rows in blocks, made once (mem holds
// half_base_bytes); whether a row is not finite can be read from scal[kScalBad] afterwards.
constexpr uint32_t kSampleShiftMin = 3, kSampleShiftMax = 6;
struct HalfBase {
    uint32_t n = 0, dim = 0, ks = 0, frags = 0, last_block = 0;
    bool ip = false;
    uint4* blocks = nullptr;  // the rows; from block sample_first[s] on one row of 2^s
    uint32_t sample_first[kSampleShiftMax + 1] = {};
    uint32_t last_sample_block = 0;
    float* centre = nullptr;
    uint32_t* scal = nullptr;
};
// whether the values that a query's bound is taken from stand for an interval so wide
bool half_scan_takes(uint64_t widest);
size_t half_base_bytes(size_t n, uint32_t dim);
int half_base_async(const float* data, size_t n, uint32_t dim, int metric, void* mem, HalfBase* out, hipStream_t st);
// One call.  Tile-grid rows as ScanRows has them (128 a row tile; row r stands for query row_query[r] and the columns [row_lo,
// row_hi)), on the device, with each query's rows (list_off, lists); on the host per row tile its column tiles of 128 and the
// mean width of its rows.
struct HalfScan {
    uint32_t rows = 0, nq = 0, k = 0;
    const uint32_t* tile_lo = nullptr;
    const uint32_t* tile_hi = nullptr;
    std::vector<uint32_t> words;  // the device tables that half_scan_plan makes, for the caller's upload
    size_t at_sweep = 0, at_sample = 0, at_tiles = 0;
    uint32_t sweep_items = 0, sample_items = 0;
    size_t sample_floats = 0, workspace_bytes = 0;
};
// false: it would need more device memory than max_bytes
bool half_scan_plan(const HalfBase& b, uint32_t num_cu, const uint32_t* h_row_lo, const uint32_t* h_row_hi, size_t max_bytes, HalfScan* s);
// everything queued on `st`: results, and (*left)[0]: whether some query is one that this way does not take (nothing of the
// results is to be used then), (*left)[1]: the number of queries not proven, from (*left)[2] on: which
struct HalfScanArgs {
    const float* data;
    const float* queries;
    const uint32_t* row_query;
    const uint32_t* row_lo;
    const uint32_t* row_hi;
    const uint32_t* list_off;
    const uint32_t* lists;
    const uint32_t* words;  // HalfScan::words on the device
    int64_t* out_ids;
    float* out_dist;
    hipEvent_t contraction_done;  // optional: recorded behind the sweep
    uint32_t* flag;               // (these two are half_scan_async's)
    uint32_t* doubt;
};
int half_scan_async(const HalfBase& b, const HalfScan& s, const HalfScanArgs& a, void* workspace, uint32_t num_cu, uint32_t** left, hipStream_t st);

// matrix work and redone rows of the calling thread's last exact_topk / scan (grab_last_knn_stats and its kin)
struct KnnStats {
    double flop = 0.0;          // fp32 matrix instructions
    double flop_bf16 = 0.0;     // half-precision matrix instructions, counted as the three that a product of split rows takes
    double flop_f16 = 0.0;      // ... those of f16 rows among them, as executed
    uint64_t redone_rows = 0;   // rows the symmetric pass handed to the plain pass
    uint64_t exact_rows = 0;    // rows (queries) that their candidates did not prove and an exact pass redid
};
KnnStats& knn_stats();
bool knn_bf16_allowed();  // grab_knn_allow_bf16

}  // namespace grab
