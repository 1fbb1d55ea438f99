// common.hpp -- shared host/device definitions of the gfx950 SpTRSV library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <array>
#include <map>
#include <string>
#include <vector>

#include "sptrsv_amd.h"

namespace sptrsv {

// ---- error plumbing --------------------------------------------------------
void set_error(const std::string& msg);
int fail(int status, const std::string& msg);
int hip_fail(hipError_t e, const char* what, const char* file, int line);

#define SPT_HIP(call)                                                        \
    do {                                                                     \
        hipError_t e_ = (call);                                              \
        if (e_ != hipSuccess) return ::sptrsv::hip_fail(e_, #call, __FILE__, __LINE__); \
    } while (0)

#define SPT_TRY(call)                 \
    do {                              \
        int s_ = (call);              \
        if (s_ != SPTRSV_OK) return s_; \
    } while (0)

// ---- constants -------------------------------------------------------------
constexpr int kWave = 64;
// Readiness is carried by the published word itself: the all-ones pattern (a
// NaN payload that arithmetic never produces, see canon64/canon32) means
// "row not solved yet".  Levels use 0 (levels are >= 1).
constexpr uint64_t kUnsolved64 = ~0ull;
constexpr uint32_t kUnsolved32 = ~0u;

// ---- device memory -----------------------------------------------------------
// Carves arrays out of one allocation (an allocation costs tens of
// microseconds, its release more, and both wait): add() every array, then get().
struct Arena {
    struct Part {
        void** p;
        size_t bytes;
    };
    std::vector<Part> parts;
    size_t total = 0;
    template <class T>
    void add(T** p, size_t count) {
        const size_t bytes = (std::max<size_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
        parts.push_back({reinterpret_cast<void**>(p), bytes});
        total += bytes;
    }
    hipError_t get(void** block) {
        const hipError_t e = hipMalloc(block, total);
        if (e != hipSuccess) return e;
        char* at = static_cast<char*>(*block);
        for (const Part& q : parts) {
            *q.p = at;
            at += q.bytes;
        }
        return e;
    }
};

// ---- library-private state hung off sp_mat_t::priv ------------------------
struct Workspace;  // defined in solve.hip

// Row tiles of the Jacobi passes: 4 ints per tile (first row, end row, first
// entry, end entry) and, for a batch, the member of each tile (device).
struct TileTable {
    int* tiles = nullptr;
    int* member = nullptr;   // null: one member
    int count = 0;
    int K = 0;               // right-hand-side width the tiles were cut for
    int rows_max = 0;        // most rows in one tile
    // entries of each tile sorted by column (built on request): column,
    // scaled value, position inside the tile (packed above the column's
    // cbits bits of sja when cbits > 0; else in sslot)
    int* sja = nullptr;
    float* ssv = nullptr;
    unsigned short* sslot = nullptr;
    int cbits = 0;
};

// Plan of the level walk (level_walk.hip) for one analysis: steps and slices,
// their slots (dependency, and the entry the value comes from), and room for the
// records, b and x of one solve, whichever precision it has.
struct LevelPlan {
    bool bad = false;            // the walk is not taken for this analysis
    bool far = false;            // entries beyond the LDS ring
    bool permuted = false;       // b and x pass through position order
    int nw = 0, nsteps = 0, n_steps_all = 0, n_slices = 0, n_over = 0;
    void* slice = nullptr;
    void* step = nullptr;
    unsigned *col = nullptr, *fcol = nullptr, *ocol = nullptr;  // slots, far slots, overflow slots
    int *from = nullptr, *ffrom = nullptr, *ofrom = nullptr;
    int* over = nullptr;         // first overflow unit of each slice
    int* diag_from = nullptr;    // entry of each position's diagonal
    int* order = nullptr;        // row of each position
    // written by every solve
    unsigned *rec = nullptr, *frec = nullptr, *orec = nullptr, *rows = nullptr;
    float* piv32 = nullptr;
    uint64_t* pub = nullptr;     // published words (mixed, far entries)
    double *b = nullptr, *x = nullptr;
    void* block = nullptr;       // the allocation that holds the arrays above
};

constexpr int kCounterWords = 16;

struct MatPriv {
    void* block = nullptr;       // holds ia, ja, a, a32 and src_perm of a handle made on the device
    int* counters = nullptr;     // [0] ticket, [1] watchdog word, [4] to [7], [9], [13] row shape, [8] XCD of a walk, [10], [11] analysis, [12] batch (device)
    uint64_t* pub = nullptr;     // published words, n*k 64-bit (device)
    size_t pub_words = 0;
    uint64_t* part = nullptr;    // published partial sums of long-row segments, 2 per segment (device)
    size_t part_words = 0;
    // level-ordered copy (config reorder = 1): this matrix with its rows in the
    // level order of an analysis, that copy's own analysis, and the caller's
    // row of each copied row; built on first use, for the analysis whose id
    // is lc_src (rebuilt for another), dropped when the values change
    sp_mat_t* lc_mat = nullptr;
    dfr_analysis_info_t* lc_info = nullptr;
    int* lc_rows = nullptr;
    unsigned long long lc_src = 0;
    std::map<unsigned long long, LevelPlan> lw;  // level walk: plan per analysis (by its id)
    // in-degree walk: per-row counters and the off-diagonal pattern by column
    // (built on first use; structure only, so new values keep them)
    int* indeg = nullptr;
    int* dep_ptr = nullptr;
    int* dep_row = nullptr;
    double* resid = nullptr;     // two-pass refinement buffers (device)
    float* corr = nullptr;
    float* b32 = nullptr;
    size_t resid_len = 0;
    long long watchdog_ticks = 0;  // wall-clock ticks a wait may last
    double wall_rate_khz = 100000.0;
    int device = 0;
    int max_row = 0;             // longest row (entries incl. diagonal)
    bool banded = false;         // no column more than 63 rows back, none twice in a row
    int band_levels = 0;         // banded: number of levels (0: not counted)
    bool most_wait = false;      // at least half of the rows have an off-diagonal
    bool many_long = false;      // more than one row in 200 has over kLongRow off-diagonals
    double nearest = 0.0;        // mean distance of the nearest off-diagonal, of the rows that have one
    bool near_rows = false;      // at least half of the rows depend on one of the kNear rows before them
    long long* trace = nullptr;  // per-row timeline (profiling), 3*n*k
    size_t trace_len = 0;
    int backoff = 0;
    unsigned lds_pad = 0;        // extra LDS per workgroup, caps resident waves
    // JACOBI refinement
    double tol = 1e-10;          // certified relative accuracy
    double margin = 0.0;         // min_i |L_ii| - sum_j |L_ij|
    bool margin_known = false;
    // upper-triangular matrix stored as the lower triangle of the reversed
    // index order: solves reverse b into rev_b and the result back from rev_x
    bool reversed = false;
    // stored entry q holds value src_perm[q] of the value array the handle
    // was created from (src_count entries; identity when src_perm is null;
    // -1 marks the constant 1.0 of a unit diagonal): sptrsv_update_values
    // gathers new values through it, keeping structure and analysis
    int* src_perm = nullptr;
    long long src_count = 0;
    void* rev_b = nullptr;
    void* rev_x = nullptr;
    size_t rev_bytes = 0;
    float* jac_r = nullptr;      // FP32 row-scaled residual D^-1 r, n*k
    float* jac_sval = nullptr;   // FP32 a_ij / a_ii (0 on the diagonal), nnz
    double* jac_diag = nullptr;  // a_ii, n (contiguous, for the first iterate)
    float* jac_a = nullptr;      // Jacobi iterates (ping-pong), n*k each
    float* jac_b = nullptr;
    size_t jac_len = 0;
    unsigned long long* jac_norms = nullptr;  // per (member, column) max |r|, max |x| (double bits), replicated
    size_t jac_norms_len = 0;    // in 64-bit words
    TileTable jac_tt[2];         // row tiles of 1024 / 2048 products (residual uses [0])
    bool jac_tiles_fixed = false;  // tiles installed by the caller (batch), never rebuilt
    int jac_members = 1;         // independent systems sharing the certificate (batch)
    // captured solves (sptrsv_solve_graph): key = precision, b, x, n, k,
    // refinement steps and the resolved configuration
    std::map<std::array<long long, 21>, hipGraphExec_t> graphs;
    hipStream_t cap_stream = nullptr;
    bool tuned[3] = {false, false, false};
    sptrsv_config_t tuned_cfg[3] = {};
    int tuned_k[3] = {0, 0, 0};
};

// Long-row segments of an analysis (its wave64 multirow layout).  A row of
// more than kSegMin off-diagonal entries keeps its first kSegOwn entries;
// the rest is cut into runs of kSegEntries, each a segment item: one wave
// folds the run in a fixed order and publishes the partial sum, and the row
// adds its partials in segment order.  The multirow walks go through
// items[] (wave w >= 0, segment g as -(g + 1)); the segments of a wave's rows
// come right before that wave, so an item only ever waits on lower items.
// The arrays live on the device.
constexpr int kSegMin = 256;
constexpr int kSegOwn = 128;
constexpr int kSegEntries = 256;
// Segments of a row with `off` off-diagonal entries.
__host__ __device__ constexpr int seg_count(int off) {
    return off > kSegMin ? (off - kSegOwn + kSegEntries - 1) / kSegEntries : 0;
}
// Published partial words: all-ones = not yet published; the poison pattern
// (NaN in every policy's view) stands in for a partial the watchdog gave up on.
constexpr uint64_t kPartPoison = 0x7ff800007fc00000ull;
struct SegTable {
    int n_items = 0;         // n_waves + n_segs
    int n_segs = 0;
    int n_split = 0;         // rows that own segments
    int* items = nullptr;    // [n_items]
    int* seg_lo = nullptr;   // first entry of each segment [n_segs]
    int* seg_hi = nullptr;   // end entry of each segment [n_segs]
    int* row_seg = nullptr;  // first segment of each row, -1 for none [n]
};
// The analysis's segment table, or null when it has none.
const SegTable* segments_of(const dfr_analysis_info_t* info);
int build_segments(dfr_analysis_info_t* info, sp_mat_t* m);
// The wave64 layout of an analysis, whatever its mode (base null: none).
struct PackedWaves {
    const int* base = nullptr;
    const int* size = nullptr;
    int n = 0;
};
PackedWaves packed_waves(const dfr_analysis_info_t* info);
// Identifies an analysis for the captured-solve cache: unique per analysis
// built, loaded or copied (never reused); 0 for none.
unsigned long long analysis_id(const dfr_analysis_info_t* info);

MatPriv* priv_of(sp_mat_t* m);
int ensure_priv(sp_mat_t* m);
// Destroys every captured solve of the matrix.  A captured solve holds the
// device addresses of the workspaces and the launch arguments it was
// captured with, so this runs before any of them is freed, reallocated or
// changed (waits for the device first: a replay may still be running).
void drop_graphs(MatPriv* pv);
void free_mat(sp_mat_t* m);  // device arrays and private state; zeroes *m
// Releases a matrix's level-ordered copy (if any).
void drop_level_copy(MatPriv* pv);
// Level walk: whether its rule takes this matrix and analysis, whether they have
// a plan (the walk is then the default shape of an analysed solve), making it
// where the rule says so, and its release.
bool level_walk_fits(const sp_mat_t* m, const dfr_analysis_info_t* info);
bool level_plan_made(const sp_mat_t* m, const dfr_analysis_info_t* info);
// (work: level_plan_work words, or null)
int make_level_plan(sp_mat_t* m, const dfr_analysis_info_t* info, int* work);
size_t level_plan_work(int nlevs);
void drop_level_plans(MatPriv* pv);
void drop_level_plan(MatPriv* pv, unsigned long long id);
// multirow_analysis_base_GPU, without the level walk's plan unless asked for.
int level_analysis(dfr_analysis_info_t** info, sp_mat_t* m, MODE mode, bool plan);
// Releases what the live matrices keep for the analysis with this id.
void analysis_freed(unsigned long long id);
// What the rows of a matrix look like, for the choice of a walk.
constexpr int kNear = 8, kLongRow = 64;
constexpr double kNoneNear = 1e30;  // nearest off-diagonal where no row has one
struct RowShape {
    int longest = 0;        // entries, with the diagonal
    bool wide = false;      // a column 64 or more rows back
    bool twice = false;     // while !wide: a row with the same column twice
    int levels = 0;         // while !wide; 0: not counted
    // for the banded kernel, which keeps one coefficient per column
    bool banded() const { return !wide && !twice; }
    long long near = 0;     // rows whose nearest off-diagonal is at most kNear rows back
    long long long_rows = 0;  // rows of more than kLongRow off-diagonals
    long long waiting = 0;  // rows with an off-diagonal
    long long dist = 0;     // sum of their distances to the nearest
    // of the `seen` rows that near, long_rows, waiting and dist were counted over
    // the same of a matrix followed by another, on the diagonal
    void add(const RowShape& o) {
        longest = std::max(longest, o.longest);
        wide |= o.wide;
        twice |= o.twice;
        levels = std::max(levels, o.levels);
        near += o.near;
        long_rows += o.long_rows;
        waiting += o.waiting;
        dist += o.dist;
    }
    void install(MatPriv* pv, long long rows, long long seen) const {
        pv->max_row = longest;
        pv->banded = banded() && rows > 0;
        pv->band_levels = banded() ? levels : 0;
        pv->near_rows = seen > 0 && 2 * near >= seen;
        pv->many_long = 200 * long_rows > seen;
        pv->most_wait = 2 * waiting >= seen;
        pv->nearest = waiting > 0 ? (double)dist / (double)waiting : kNoneNear;
    }
};
// The same of a matrix made on the device (its longest row given; waits).
int install_row_shape(sp_mat_t* m, int longest);
// Whether the block walk is the default of a natural-order solve, and whether
// it takes its rows in order (banded kernel).
bool block_walk_fits(const sp_mat_t* m);
bool block_walk_in_order(const sp_mat_t* m);
// Banded with less than four rows per level: the block walk, analysed or not.
bool chain_of(const sp_mat_t* m, const dfr_analysis_info_t* info);
// Lanes per row of the group walk where that is the natural-order default, else 0.
int group_walk_lanes(const sp_mat_t* m);
// Rows per level below which a banded matrix is taken in order.
constexpr long long kBandRows = 16;
void free_info_arrays(dfr_analysis_info_t* info);
// The analysis of `copy`, the level-ordered copy made for analysis `src`,
// derived from `src` (levels permuted, iorder the identity, the rest shared).
int level_copy_analysis(const dfr_analysis_info_t* src, sp_mat_t* copy, dfr_analysis_info_t* dst);

// out[i] = sum_{j<i} in[j] on the device (in and out may alias)
// With scratch (scan_scratch(n) ints) it only launches; else it allocates and
// waits.
int exclusive_scan(const int* in, int* out, long long n, hipStream_t s, int* scratch = nullptr);
size_t scan_scratch(long long n);
// Kernel timer (api_solve.hip): the next (start, stop) event pair while
// timing is enabled and the stream is not being captured, else an empty
// pair (false); the caller records it around `launches` consecutive
// launches of one kernel.  Returned by value: the pool may grow meanwhile.
struct KtPair {
    hipEvent_t ev[2] = {nullptr, nullptr};
    explicit operator bool() const { return ev[0] != nullptr; }
    hipEvent_t operator[](int i) const { return ev[i]; }
};
constexpr int kTimeSyncFree = 1;   // sync-free solve passes (kernel timer kinds)
constexpr int kTimeSweeps = 2;     // a refinement step's Jacobi sweeps
KtPair kernel_timer_pair(hipStream_t s, int launches = 1, int kind = kTimeSyncFree);
// stable LSD radix sort of (keys, vals) by key in [0, max_key]; tk/tv scratch
// (with sort_scratch(n) ints of scratch it only launches).
int radix_sort_pairs(int* keys, int* vals, int* tk, int* tv, int n, int max_key, hipStream_t s, int* scratch = nullptr);
size_t sort_scratch(int n);
// Longest row of a device row-pointer array into out[0], rows of more than
// kLongRow off-diagonals into out[1] (device, zero before).
int longest_row(const int* ia, int n, int* out, hipStream_t s);

// ---- launch helpers ----------------------------------------------------------
inline unsigned ceil_div(long long a, long long b) { return (unsigned)((a + b - 1) / b); }

}  // namespace sptrsv
