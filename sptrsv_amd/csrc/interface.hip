// interface.hip -- host interface (interface.h:6-9 / interface.cu:9-102),
// error reporting, device helpers and the BENCH_RUN_SOLVE equivalent
// (common.h:103-124).
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <unordered_set>
#include <vector>

#include "common.hpp"

namespace sptrsv {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }

int fail(int status, const std::string& msg) {
    g_last_error = msg;
    return status;
}

int hip_fail(hipError_t e, const char* what, const char* file, int line) {
    std::string m = std::string(what) + ": " + hipGetErrorString(e) + " (" + file + ":" +
                    std::to_string(line) + ")";
    g_last_error = m;
    if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) return SPTRSV_E_ALLOC;
    return SPTRSV_E_HIP;
}

MatPriv* priv_of(sp_mat_t* m) { return static_cast<MatPriv*>(m->priv); }

// Handles alive in this process, so that the library's teardown can release
// the HIP objects of handles their owners never freed.
static std::mutex g_live_mu;
static std::unordered_set<MatPriv*> g_live;

void drop_graphs(MatPriv* pv) {
    if (!pv || pv->graphs.empty()) return;
    (void)hipDeviceSynchronize();
    for (auto& g : pv->graphs) (void)hipGraphExecDestroy(g.second);
    pv->graphs.clear();
}

void analysis_freed(unsigned long long id) {
    std::lock_guard<std::mutex> g(g_live_mu);
    for (MatPriv* pv : g_live) drop_level_plan(pv, id);
}

int convert_values_to_f32(sp_mat_t* m);
void free_info_arrays(dfr_analysis_info_t* info);
int jacobi_values_changed(sp_mat_t* m);

// a[q] (and a32[q]) = src[perm[q]]; identity map when perm is null, the
// constant 1.0 where perm[q] < 0.
template <bool F64>
__global__ void k_gather_values(const int* __restrict__ perm, const double* __restrict__ src, int nnz,
                                double* __restrict__ a, float* __restrict__ a32) {
    for (long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x; q < nnz;
         q += (long long)gridDim.x * blockDim.x) {
        const int p = perm ? perm[q] : (int)q;
        const double v = p >= 0 ? src[p] : 1.0;
        if constexpr (F64) a[q] = v;
        a32[q] = (float)v;
    }
}

static double watchdog_ms_default() {
    const char* e = getenv("SPTRSV_WATCHDOG_MS");
    if (e) {
        double v = atof(e);
        if (v > 0) return v;
    }
    return 20000.0;
}

int ensure_priv(sp_mat_t* m) {
    if (m->priv) return SPTRSV_OK;
    MatPriv* pv = new MatPriv();
    SPT_HIP(hipGetDevice(&pv->device));
    int rate = 0;
    if (hipDeviceGetAttribute(&rate, hipDeviceAttributeWallClockRate, pv->device) == hipSuccess &&
        rate > 0)
        pv->wall_rate_khz = rate;
    pv->watchdog_ticks = (long long)(watchdog_ms_default() * pv->wall_rate_khz);
    hipError_t e = hipMalloc(&pv->counters, kCounterWords * sizeof(int));
    if (e != hipSuccess) {
        delete pv;
        return hip_fail(e, "hipMalloc counters", __FILE__, __LINE__);
    }
    SPT_HIP(hipMemset(pv->counters, 0, kCounterWords * sizeof(int)));
    m->priv = pv;
    std::lock_guard<std::mutex> g(g_live_mu);
    g_live.insert(pv);
    return SPTRSV_OK;
}

void free_mat(sp_mat_t* m) {
    if (!m) return;
    MatPriv* pv = priv_of(m);
    if (pv && pv->block) {
        (void)hipFree(pv->block);
        pv->src_perm = nullptr;
    } else {
        if (m->ia) (void)hipFree(m->ia);
        if (m->ja) (void)hipFree(m->ja);
        if (m->a) (void)hipFree(m->a);
        if (m->a32) (void)hipFree(m->a32);
    }
    if (pv) {
        {
            // first, so that no freed analysis looks at this matrix any more
            std::lock_guard<std::mutex> g(g_live_mu);
            g_live.erase(pv);
        }
        drop_level_copy(pv);
        drop_level_plans(pv);
        if (pv->counters) (void)hipFree(pv->counters);
        if (pv->pub) (void)hipFree(pv->pub);
        if (pv->part) (void)hipFree(pv->part);
        for (int* q : {pv->indeg, pv->dep_ptr, pv->dep_row})
            if (q) (void)hipFree(q);
        if (pv->b32) (void)hipFree(pv->b32);
        if (pv->corr) (void)hipFree(pv->corr);
        if (pv->resid) (void)hipFree(pv->resid);
        if (pv->trace) (void)hipFree(pv->trace);
        if (pv->src_perm) (void)hipFree(pv->src_perm);
        if (pv->rev_b) (void)hipFree(pv->rev_b);
        if (pv->rev_x) (void)hipFree(pv->rev_x);
        for (float* p : {pv->jac_r, pv->jac_a, pv->jac_b, pv->jac_sval})
            if (p) (void)hipFree(p);
        if (pv->jac_diag) (void)hipFree(pv->jac_diag);
        if (pv->jac_norms) (void)hipFree(pv->jac_norms);
        for (auto& g : pv->graphs) (void)hipGraphExecDestroy(g.second);
        if (pv->cap_stream) (void)hipStreamDestroy(pv->cap_stream);
        for (TileTable& t : pv->jac_tt) {
            if (t.tiles) (void)hipFree(t.tiles);
            if (t.member) (void)hipFree(t.member);
            if (t.sja) (void)hipFree(t.sja);
            if (t.ssv) (void)hipFree(t.ssv);
            if (t.sslot) (void)hipFree(t.sslot);
        }
        delete pv;
    }
    memset(m, 0, sizeof(*m));
}

// out[0] bit 1: a column 64 or more rows back, 2: a row with a column twice
// (counted where bit 1 is not set); out[1]: rows whose nearest off-diagonal is at
// most kNear rows back; out[5]: rows of more than kLongRow off-diagonals; out[9]:
// rows with an off-diagonal; dist: the sum of their distances.  Columns may come in any order, so all are read,
// eight lanes a row; few workgroups, large ones, as each adds to the same words
// (2D grid 250^2 from coordinates: 573 -> 510 us from 2048 workgroups of 256 threads).
constexpr int kShapeLanes = 8, kShapeThreads = 1024;
__global__ __launch_bounds__(kShapeThreads) void k_row_shape(const int* __restrict__ ia, const int* __restrict__ ja, int n,
                                                   int* __restrict__ out, unsigned long long* __restrict__ dist) {
    __shared__ int s_near, s_flags, s_long, s_waiting;
    __shared__ unsigned long long s_dist;
    if (threadIdx.x == 0) {
        s_near = s_flags = s_long = s_waiting = 0;
        s_dist = 0;
    }
    __syncthreads();
    int near = 0, flags = 0, longer = 0, waiting = 0;
    unsigned long long far = 0;
    const int e = threadIdx.x % kShapeLanes;
    const long long rows = (long long)gridDim.x * blockDim.x / kShapeLanes;
    // (whole groups of lanes enter and leave together)
    for (long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / kShapeLanes; i < n; i += rows) {
        const int lo = ia[i], hi = ia[i + 1] - 1;
        int least = 0x7fffffff;
        unsigned long long seen = 0;  // distances of this lane's entries
        for (int p = lo + e; p < hi; p += kShapeLanes) {
            const int d = (int)i - ja[p];
            least = min(least, d);
            if (d >= kWave) {
                flags |= 1;
            } else {
                flags |= (seen >> d) & 1 ? 2 : 0;
                seen |= 1ull << d;
            }
        }
        for (int o = 1; o < kShapeLanes; o <<= 1) {
            least = min(least, __shfl_xor(least, o));
            const unsigned long long other = __shfl_xor(seen, o);
            flags |= seen & other ? 2 : 0;
            seen |= other;
        }
        if (e == 0 && lo < hi) {
            near += least <= kNear;
            far += least;
            ++waiting;
            longer += hi - lo > kLongRow;
        }
    }
    if (near) atomicAdd(&s_near, near);
    if (far) atomicAdd(&s_dist, far);
    if (longer) atomicAdd(&s_long, longer);
    if (flags) atomicOr(&s_flags, flags);
    if (waiting) atomicAdd(&s_waiting, waiting);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_flags) atomicOr(&out[0], s_flags);
        if (s_near) atomicAdd(&out[1], s_near);
        if (s_dist) atomicAdd(dist, s_dist);
        if (s_long) atomicAdd(&out[5], s_long);
        if (s_waiting) atomicAdd(&out[9], s_waiting);
    }
}

int install_row_shape(sp_mat_t* m, int longest) {
    RowShape shape;
    shape.longest = longest;
    const int n = m->nr;
    if (n > 0) {
        int h[10] = {}, *d = priv_of(m)->counters + 4;  // zero since the handle was made
        hipLaunchKernelGGL(k_row_shape, dim3(std::min<unsigned>(ceil_div((long long)n * kShapeLanes, kShapeThreads), 256)), dim3(kShapeThreads), 0, nullptr, m->ia,
                           m->ja, n, d, reinterpret_cast<unsigned long long*>(d + 2));
        SPT_HIP(hipGetLastError());
        SPT_HIP(hipMemcpy(h, d, sizeof(h), hipMemcpyDeviceToHost));
        shape.wide = (h[0] & 1) != 0;
        shape.twice = (h[0] & 2) != 0;
        shape.near = h[1];
        shape.long_rows = h[5];
        shape.waiting = h[9];
        memcpy(&shape.dist, h + 2, sizeof(shape.dist));
    }
    shape.install(priv_of(m), n, n);
    return SPTRSV_OK;
}

// Validates a host CSR lower triangle: every row non-empty, diagonal last,
// off-diagonal columns in [0, i).  Adds its rows to *shape.
static int validate_host_csr(const int* ia, const int* ja, int n, RowShape* shape) {
    if (n < 0) return fail(SPTRSV_E_INVALID_ARG, "n < 0");
    if (n == 0) return SPTRSV_OK;
    if (!ia || !ja) return fail(SPTRSV_E_INVALID_ARG, "null CSR arrays");
    const int base = ia[0];
    if (base < 0) return fail(SPTRSV_E_INVALID_CSR, "negative row pointer");
    ja += base;  // rows index ja relative to ia[0]
    int lev[kWave] = {};   // levels of the last 64 rows, while they are all that is needed
    int seen[kWave] = {};  // row + 1 that last had a column, likewise
    for (int i = 0; i < n; ++i) {
        int level = 1, nearest = -1;
        long long s = (long long)ia[i] - base, e = (long long)ia[i + 1] - base;
        if (e <= s)
            return fail(SPTRSV_E_INVALID_CSR, "row " + std::to_string(i) + " has no diagonal entry");
        if (ja[e - 1] != i)
            return fail(SPTRSV_E_INVALID_CSR,
                        "row " + std::to_string(i) + ": last entry is not the diagonal");
        for (long long p = s; p < e - 1; ++p) {
            if (ja[p] < 0 || ja[p] >= i)
                return fail(SPTRSV_E_INVALID_CSR, "row " + std::to_string(i) + ": column " +
                                                      std::to_string(ja[p]) +
                                                      " outside the strict lower triangle");
            shape->wide |= i - ja[p] >= kWave;
            nearest = std::max(nearest, ja[p]);  // (columns in any order)
            if (shape->wide) continue;
            level = std::max(level, lev[ja[p] % kWave] + 1);
            int& s = seen[ja[p] % kWave];
            shape->twice |= s == i + 1;
            s = i + 1;
        }
        lev[i % kWave] = level;
        shape->levels = std::max(shape->levels, level);
        if (e - s > 1) {
            shape->near += i - nearest <= kNear;
            shape->dist += i - nearest;
            ++shape->waiting;
        }
        shape->longest = std::max<int>(shape->longest, (int)(e - s));
        shape->long_rows += e - s > kLongRow + 1;
    }
    return SPTRSV_OK;
}

template <class V>
static int upload(const int* ia, const int* ja, const V* val, int n, sp_mat_t* m) {
    if (!m) return fail(SPTRSV_E_INVALID_ARG, "null sp_mat_t");
    RowShape shape;
    memset(m, 0, sizeof(*m));
    SPT_TRY(validate_host_csr(ia, ja, n, &shape));
    if (n > 0 && !val) return fail(SPTRSV_E_INVALID_ARG, "null values");
    long long nnz = n > 0 ? (long long)ia[n] - ia[0] : 0;
    if (nnz > 0x7fffffffLL) return fail(SPTRSV_E_CAPACITY, "nnz exceeds int32");
    SPT_TRY(ensure_priv(m));
    shape.install(priv_of(m), n, n);
    m->nr = n;
    m->nc = n;
    m->nnz = (int)nnz;
    std::vector<int> rebased;
    const int* ia_up = ia;
    if (n > 0 && ia[0] != 0) {
        rebased.resize(n + 1);
        for (int i = 0; i <= n; ++i) rebased[i] = ia[i] - ia[0];
        ia_up = rebased.data();
    }
    const size_t off = n > 0 ? (size_t)ia[0] : 0;
    int st = SPTRSV_OK;
    auto chk = [&](hipError_t e, const char* what) {
        if (e != hipSuccess && st == SPTRSV_OK) st = hip_fail(e, what, __FILE__, __LINE__);
    };
    chk(hipMalloc(&m->ia, sizeof(int) * (size_t)(n + 1)), "hipMalloc ia");
    chk(hipMalloc(&m->ja, sizeof(int) * (size_t)std::max<long long>(nnz, 1)), "hipMalloc ja");
    chk(hipMalloc(&m->a32, sizeof(float) * (size_t)std::max<long long>(nnz, 1)), "hipMalloc a32");
    if (st == SPTRSV_OK && n == 0) chk(hipMemset(m->ia, 0, sizeof(int)), "memset ia");
    if (st == SPTRSV_OK && n > 0) {
        chk(hipMemcpy(m->ia, ia_up, sizeof(int) * (size_t)(n + 1), hipMemcpyHostToDevice), "copy ia");
        chk(hipMemcpy(m->ja, ja + off, sizeof(int) * (size_t)nnz, hipMemcpyHostToDevice), "copy ja");
    }
    if (st == SPTRSV_OK) {
        if constexpr (sizeof(V) == 8) {
            chk(hipMalloc(&m->a, sizeof(double) * (size_t)std::max<long long>(nnz, 1)), "hipMalloc a");
            if (st == SPTRSV_OK && nnz > 0)
                chk(hipMemcpy(m->a, val + off, sizeof(double) * (size_t)nnz, hipMemcpyHostToDevice),
                    "copy a");
            if (st == SPTRSV_OK) st = convert_values_to_f32(m);
        } else {
            if (nnz > 0)
                chk(hipMemcpy(m->a32, val + off, sizeof(float) * (size_t)nnz, hipMemcpyHostToDevice),
                    "copy a32");
        }
    }
    if (st == SPTRSV_OK) chk(hipDeviceSynchronize(), "upload sync");
    if (st == SPTRSV_OK) priv_of(m)->src_count = nnz;
    if (st != SPTRSV_OK) free_mat(m);
    return st;
}


// Plain streaming copy, 16 bytes per thread and step: the reference kernel
// for scaling hardware traffic counters (reads n*16 bytes, writes n*16).
static __global__ void k_copy16(uint4* __restrict__ dst, const uint4* __restrict__ src, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

static __global__ void k_add_offset(int* p, size_t count, int off) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (size_t)gridDim.x * blockDim.x)
        p[i] += off;
}

static unsigned add_grid(size_t count) {
    size_t g = (count + 255) / 256;
    return (unsigned)std::max<size_t>(1, std::min<size_t>(g, 8192));
}

// Uploads nmat host CSR lower triangles as one block-diagonal matrix with
// global row and column indices; row_off receives the first row of each.
int upload_concat(const int* n, const int* const* ia, const int* const* ja, const double* const* a,
                  int nmat, sp_mat_t* m, std::vector<long long>& row_off, std::vector<RowShape>* shapes) {
    memset(m, 0, sizeof(*m));
    row_off.assign(nmat + 1, 0);
    std::vector<long long> nnz_off(nmat + 1, 0);
    RowShape shape;
    for (int q = 0; q < nmat; ++q) {
        if (n[q] < 0) return fail(SPTRSV_E_INVALID_ARG, "negative size");
        RowShape own;
        int st = validate_host_csr(ia[q], ja[q], n[q], &own);
        if (st != SPTRSV_OK) return fail(st, "matrix " + std::to_string(q) + ": " + g_last_error);
        shapes->push_back(own);
        shape.add(own);
        row_off[q + 1] = row_off[q] + n[q];
        nnz_off[q + 1] = nnz_off[q] + (n[q] > 0 ? (long long)ia[q][n[q]] - ia[q][0] : 0);
    }
    const long long rows = row_off[nmat], nnz = nnz_off[nmat];
    if (rows > 0x7ffffffeLL || nnz > 0x7fffffffLL) return fail(SPTRSV_E_CAPACITY, "batch exceeds int32 indexing");
    SPT_TRY(ensure_priv(m));
    shape.install(priv_of(m), rows, rows);
    m->nr = m->nc = (int)rows;
    m->nnz = (int)nnz;
    int st = SPTRSV_OK;
    auto chk = [&](hipError_t e, const char* what) {
        if (e != hipSuccess && st == SPTRSV_OK) st = hip_fail(e, what, __FILE__, __LINE__);
    };
    chk(hipMalloc(&m->ia, sizeof(int) * (size_t)(rows + 1)), "hipMalloc ia");
    chk(hipMalloc(&m->ja, sizeof(int) * (size_t)std::max<long long>(nnz, 1)), "hipMalloc ja");
    chk(hipMalloc(&m->a, sizeof(double) * (size_t)std::max<long long>(nnz, 1)), "hipMalloc a");
    chk(hipMalloc(&m->a32, sizeof(float) * (size_t)std::max<long long>(nnz, 1)), "hipMalloc a32");
    for (int q = 0; q < nmat && st == SPTRSV_OK; ++q) {
        if (n[q] == 0) continue;
        const size_t nz = (size_t)(nnz_off[q + 1] - nnz_off[q]);
        const size_t b0 = (size_t)ia[q][0];
        chk(hipMemcpy(m->ia + row_off[q], ia[q], sizeof(int) * (size_t)n[q], hipMemcpyHostToDevice), "copy ia");
        chk(hipMemcpy(m->ja + nnz_off[q], ja[q] + b0, sizeof(int) * nz, hipMemcpyHostToDevice), "copy ja");
        chk(hipMemcpy(m->a + nnz_off[q], a[q] + b0, sizeof(double) * nz, hipMemcpyHostToDevice), "copy a");
        if (st != SPTRSV_OK) break;
        hipLaunchKernelGGL(k_add_offset, dim3(add_grid((size_t)n[q])), dim3(256), 0, nullptr,
                           m->ia + row_off[q], (size_t)n[q], (int)(nnz_off[q] - ia[q][0]));
        hipLaunchKernelGGL(k_add_offset, dim3(add_grid(nz)), dim3(256), 0, nullptr, m->ja + nnz_off[q], nz,
                           (int)row_off[q]);
        chk(hipGetLastError(), "offset kernels");
    }
    if (st == SPTRSV_OK) {
        int last = (int)nnz;
        chk(hipMemcpy(m->ia + rows, &last, sizeof(int), hipMemcpyHostToDevice), "copy ia end");
    }
    if (st == SPTRSV_OK) st = convert_values_to_f32(m);
    if (st == SPTRSV_OK) chk(hipDeviceSynchronize(), "upload sync");
    if (st != SPTRSV_OK) free_mat(m);
    return st;
}


// ---- dependency latency probe ------------------------------------------------------
// Block 0 and block `partner` (placed on another XCD by the round-robin
// dispatch) hand a counter back and forth through agent-scope relaxed
// stores and polling loads, the primitives of the sync-free solves.  Every
// wait is bounded; out[0..1] = elapsed wall-clock ticks, out[2] = error.
static __global__ void k_pingpong(unsigned* flags, int partner, int rounds, long long* out, int max_spin) {
    const int b = blockIdx.x;
    if ((b != 0 && b != partner) || threadIdx.x != 0) return;
    unsigned* mine = flags + (b == 0 ? 0 : 32);
    unsigned* other = flags + (b == 0 ? 32 : 0);
    long long t0 = wall_clock64();
    int err = 0;
    for (int i = 0; i < rounds && !err; ++i) {
        unsigned want = 2u * (unsigned)i + 1u;
        if (b == 0) __hip_atomic_store(mine, want, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int s = 0;
        while (__hip_atomic_load(other, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != want)
            if (++s > max_spin) { err = 1; break; }
        if (b != 0 && !err) __hip_atomic_store(mine, want, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    long long t1 = wall_clock64();
    if (b == 0) out[0] = t1 - t0;
    if (err) out[2] = 1;
}

// hip events for sptrsv_timer_*
static std::mutex g_timer_mu;
static hipEvent_t g_t0 = nullptr, g_t1 = nullptr;

}  // namespace sptrsv

using namespace sptrsv;

extern "C" {

const char* sptrsv_status_string(int status) {
    switch (status) {
        case SPTRSV_OK: return "ok";
        case SPTRSV_E_NO_ANALYSIS_NEEDED: return "SIMPLE mode needs no analysis";
        case SPTRSV_E_INVALID_ARG: return "invalid argument";
        case SPTRSV_E_INVALID_CSR: return "invalid lower-triangular CSR";
        case SPTRSV_E_ALLOC: return "device allocation failed";
        case SPTRSV_E_HIP: return "HIP runtime error";
        case SPTRSV_E_WATCHDOG: return "dependency wait exceeded its bound";
        case SPTRSV_E_NOT_ANALYSED: return "solver needs an analysis";
        case SPTRSV_E_UNAVAILABLE: return "optional runtime unavailable";
        case SPTRSV_E_IO: return "Matrix Market read error";
        case SPTRSV_E_CAPACITY: return "request exceeds a fixed capacity";
        case SPTRSV_E_NOT_CONVERGED: return "iterative solve missed its certified accuracy";
        default: return "unknown status";
    }
}

const char* sptrsv_last_error(void) { return g_last_error.c_str(); }

int allocate_memory(const int* csrRowPtrL, const int* csrColIdxL, const double* csrValL, int n,
                    sp_mat_t* gpu_L, MODE mode) {
    (void)mode;
    return upload(csrRowPtrL, csrColIdxL, csrValL, n, gpu_L);
}

int allocate_memory_f32(const int* csrRowPtrL, const int* csrColIdxL, const float* csrValL, int n,
                        sp_mat_t* gpu_L, MODE mode) {
    (void)mode;
    return upload(csrRowPtrL, csrColIdxL, csrValL, n, gpu_L);
}

// Upper triangle with the diagonal first in every row and the other columns
// in (i, n): uploaded as the lower triangle of the reversed index order,
// row n-1-i holding columns n-1-j in reversed entry order (diagonal last).
int allocate_memory_upper(const int* csrRowPtrU, const int* csrColIdxU, const double* csrValU, int n,
                          sp_mat_t* gpu_U, MODE mode) {
    (void)mode;
    if (!gpu_U) return fail(SPTRSV_E_INVALID_ARG, "null sp_mat_t");
    if (n < 0 || (n > 0 && (!csrRowPtrU || !csrColIdxU || !csrValU))) return fail(SPTRSV_E_INVALID_ARG, "null CSR");
    if (n == 0) return upload(csrRowPtrU, csrColIdxU, csrValU, n, gpu_U);
    const long long base = csrRowPtrU[0];
    if (base < 0) return fail(SPTRSV_E_INVALID_CSR, "negative row pointer");
    const long long nnz = (long long)csrRowPtrU[n] - base;
    if (nnz < n || nnz > 0x7fffffffLL) return fail(SPTRSV_E_INVALID_CSR, "bad row pointers");
    std::vector<int> ia(n + 1), ja((size_t)nnz), perm((size_t)nnz);
    std::vector<double> a((size_t)nnz);
    long long w = 0;
    ia[0] = 0;
    for (int r = 0; r < n; ++r) {
        const int i = n - 1 - r;
        const long long s = (long long)csrRowPtrU[i] - base, e = (long long)csrRowPtrU[i + 1] - base;
        if (e <= s || s < 0 || e > nnz)
            return fail(SPTRSV_E_INVALID_CSR, "row " + std::to_string(i) + " has no diagonal entry");
        if (csrColIdxU[base + s] != i)
            return fail(SPTRSV_E_INVALID_CSR, "row " + std::to_string(i) + ": first entry is not the diagonal");
        for (long long p = e - 1; p >= s; --p) {
            const int j = csrColIdxU[base + p];
            if (p > s && (j <= i || j >= n))
                return fail(SPTRSV_E_INVALID_CSR, "row " + std::to_string(i) + ": column " + std::to_string(j) +
                                                      " outside the strict upper triangle");
            ja[(size_t)w] = n - 1 - j;
            a[(size_t)w] = csrValU[base + p];
            perm[(size_t)w] = (int)p;
            ++w;
        }
        ia[r + 1] = (int)w;
    }
    SPT_TRY(upload(ia.data(), ja.data(), a.data(), n, gpu_U));
    MatPriv* pv = priv_of(gpu_U);
    pv->reversed = true;
    int st = SPTRSV_OK;
    if (hipMalloc(&pv->src_perm, sizeof(int) * (size_t)nnz) != hipSuccess ||
        hipMemcpy(pv->src_perm, perm.data(), sizeof(int) * (size_t)nnz, hipMemcpyHostToDevice) != hipSuccess)
        st = fail(SPTRSV_E_ALLOC, "value permutation");
    if (st != SPTRSV_OK) free_mat(gpu_U);
    return st;
}

void free_device_analysis(sp_mat_t* gpu_L, dfr_analysis_info_t* info) {
    if (info) free_info_arrays(info);
    if (gpu_L && gpu_L->priv) free_mat(gpu_L);
}

int sptrsv_update_values(sp_mat_t* mat, const double* vals, long long count, int on_device) {
    if (!mat || !mat->priv) return fail(SPTRSV_E_INVALID_ARG, "matrix not allocated");
    MatPriv* pv = priv_of(mat);
    if (!pv->src_perm && pv->src_count != mat->nnz)
        return fail(SPTRSV_E_INVALID_ARG, "this handle does not record where its values come from");
    if (count != pv->src_count || (count > 0 && !vals))
        return fail(SPTRSV_E_INVALID_ARG, "value count " + std::to_string(count) + " differs from the " +
                                              std::to_string(pv->src_count) + " the handle was created from");
    if (mat->nnz == 0) return SPTRSV_OK;
    const double* src = vals;
    double* staged = nullptr;
    if (!on_device && count > 0) {
        SPT_HIP(hipMalloc(&staged, sizeof(double) * (size_t)count));
        if (hipMemcpy(staged, vals, sizeof(double) * (size_t)count, hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(staged);
            return fail(SPTRSV_E_HIP, "copy values");
        }
        src = staged;
    }
    const unsigned g = (unsigned)std::max<long long>(1, std::min<long long>(16384, ((long long)mat->nnz + 255) / 256));
    if (mat->a)
        hipLaunchKernelGGL(k_gather_values<true>, dim3(g), dim3(256), 0, nullptr, pv->src_perm, src, mat->nnz,
                           mat->a, mat->a32);
    else
        hipLaunchKernelGGL(k_gather_values<false>, dim3(g), dim3(256), 0, nullptr, pv->src_perm, src, mat->nnz,
                           nullptr, mat->a32);
    int st = hipGetLastError() == hipSuccess ? SPTRSV_OK : fail(SPTRSV_E_HIP, "value gather launch");
    if (st == SPTRSV_OK && hipDeviceSynchronize() != hipSuccess) st = fail(SPTRSV_E_HIP, "value gather");
    if (staged) (void)hipFree(staged);
    SPT_TRY(st);
    // derived data: Jacobi's scaled copies and margin; captured solves bake
    // the margin into their launches, so they are dropped; a tuned Jacobi
    // choice may no longer apply (dominance can be lost)
    if (mat->a) SPT_TRY(jacobi_values_changed(mat));
    drop_level_copy(pv);  // holds the old values; rebuilt on its next use
    drop_graphs(pv);
    for (int p = 0; p < 3; ++p)
        if (pv->tuned[p] && pv->tuned_cfg[p].kernel == SPTRSV_KERNEL_JACOBI) pv->tuned[p] = false;
    return SPTRSV_OK;
}

}  // extern "C"

namespace sptrsv {

// test.h:4 / test.cu:4-30, the flow main.cu:259 runs: upload L, analyse
// (ALL), b = L * 1 summed in storage order (test.cu:13-16), then each of the
// three solvers under the BENCH_RUN_SOLVE timing (common.h:103-124, one
// repetition as BENCH_REPEAT) with the exact x == 1 check (validate_x,
// matrix_properties.h:7-29), printing one line per solver as the reference
// does.  V is VALUE_TYPE: double runs the FP64 solvers, float the FP32 ones.
// Returns the summed validate_x counts (0 = every solver passed), or a
// negative status.
template <class V>
static int test_flow(const char* filename, int* ia, int* ja, V* a, int n) {
    if (n < 0 || (n > 0 && (!ia || !ja || !a))) return fail(SPTRSV_E_INVALID_ARG, "null CSR arrays");
    constexpr bool F64 = sizeof(V) == 8;
    sp_mat_t L{};
    if constexpr (F64) SPT_TRY(allocate_memory(ia, ja, a, n, &L, ALL));
    else SPT_TRY(allocate_memory_f32(ia, ja, a, n, &L, ALL));
    dfr_analysis_info_t info{};
    info.mode = ALL;
    int st = run_analysis(&info, &L);
    std::vector<V> b((size_t)std::max(n, 1), V(0));
    for (int i = 0; i < n; ++i)
        for (int j = ia[i]; j < ia[i + 1]; ++j) b[(size_t)i] += a[j];
    V *db = nullptr, *dx = nullptr;
    if (st == SPTRSV_OK && hipMalloc(&db, sizeof(V) * b.size()) != hipSuccess) st = fail(SPTRSV_E_ALLOC, "b");
    if (st == SPTRSV_OK && hipMalloc(&dx, sizeof(V) * b.size()) != hipSuccess) st = fail(SPTRSV_E_ALLOC, "x");
    if (st == SPTRSV_OK && hipMemcpy(db, b.data(), sizeof(V) * b.size(), hipMemcpyHostToDevice) != hipSuccess)
        st = fail(SPTRSV_E_HIP, "copy b");
    if (st == SPTRSV_OK)
        printf("%s: n = %d, nnz = %d, %d levels\n", filename ? filename : "(matrix)", L.nr, L.nnz, info.nlevs);
    int errors = 0;
    const struct {
        const char* name;
        int kernel;
    } solvers[] = {{"solve base", SPTRSV_KERNEL_SIMPLE},
                   {"solve order", SPTRSV_KERNEL_ORDER},
                   {"solve multirow", SPTRSV_KERNEL_MULTIROW}};
    for (const auto& sv : solvers) {
        if (st != SPTRSV_OK || n == 0) break;
        sptrsv_config_t c{};
        c.kernel = sv.kernel;
        c.fused = 1;
        sptrsv_bench_t r{};
        st = sptrsv_bench_solve(&L, &info, F64 ? SPTRSV_PREC_F64 : SPTRSV_PREC_F32, &c, db, dx, n, 1, 1, 1, 1, &r);
        if (st != SPTRSV_OK) break;
        printf("%20.20s ----- %6.3f ms (stdev=%6.3f ms) ----- %6.2f W ----- ", sv.name, r.mean_ms, r.stdev_ms,
               r.power_mw >= 0 ? r.power_mw / 1000.0 : 0.0);
        if (r.errors) printf("[FAILED! %d errors]\n", r.errors);
        else printf("[PASS!]\n");
        errors += r.errors;
    }
    fflush(stdout);
    if (db) (void)hipFree(db);
    if (dx) (void)hipFree(dx);
    free_device_analysis(&L, &info);
    return st != SPTRSV_OK ? st : errors;
}

}  // namespace sptrsv

extern "C" {

int test_solve_L_analysis_multirow(const char* filename, int* csrRowPtrL, int* csrColIdxL, double* csrValL,
                                   int n) {
    return test_flow(filename, csrRowPtrL, csrColIdxL, csrValL, n);
}

int test_solve_L_analysis_multirow_f32(const char* filename, int* csrRowPtrL, int* csrColIdxL, float* csrValL,
                                       int n) {
    return test_flow(filename, csrRowPtrL, csrColIdxL, csrValL, n);
}

int run_solver(sp_mat_t* gpu_L, dfr_analysis_info_t* info, const double* b, double* x, int n) {
    if (!gpu_L || !gpu_L->priv) return fail(SPTRSV_E_INVALID_ARG, "matrix not allocated");
    if (n != gpu_L->nr) return fail(SPTRSV_E_INVALID_ARG, "n differs from the matrix row count");
    if (n == 0) return SPTRSV_OK;
    if (!b || !x) return fail(SPTRSV_E_INVALID_ARG, "null b or x");
    sptrsv_config_t c{SPTRSV_KERNEL_SIMPLE, 0, 0, 1};
    dfr_analysis_info_t* use = nullptr;
    if (info && info->mode != SIMPLE) {
        use = info;
        c.kernel = info->mode == ORDER ? SPTRSV_KERNEL_ORDER
                   : info->mode == MULTIROW ? SPTRSV_KERNEL_MULTIROW : SPTRSV_KERNEL_AUTO;
    }
    double *db = nullptr, *dx = nullptr;
    SPT_HIP(hipMalloc(&db, sizeof(double) * (size_t)n));
    hipError_t e = hipMalloc(&dx, sizeof(double) * (size_t)n);
    if (e != hipSuccess) {
        (void)hipFree(db);
        return hip_fail(e, "hipMalloc x", __FILE__, __LINE__);
    }
    int st = SPTRSV_OK;
    if (hipMemcpy(db, b, sizeof(double) * (size_t)n, hipMemcpyHostToDevice) != hipSuccess)
        st = fail(SPTRSV_E_HIP, "copy b");
    if (st == SPTRSV_OK) st = sptrsv_solve(gpu_L, use, SPTRSV_PREC_F64, &c, db, dx, n, 1, 1, nullptr);
    if (st == SPTRSV_OK) st = sptrsv_check(gpu_L, nullptr);
    if (st == SPTRSV_OK &&
        hipMemcpy(x, dx, sizeof(double) * (size_t)n, hipMemcpyDeviceToHost) != hipSuccess)
        st = fail(SPTRSV_E_HIP, "copy x");
    (void)hipFree(db);
    (void)hipFree(dx);
    return st;
}

// ---- device helpers -------------------------------------------------------------
int sptrsv_device_count(int* count) {
    if (!count) return fail(SPTRSV_E_INVALID_ARG, "null count");
    SPT_HIP(hipGetDeviceCount(count));
    return SPTRSV_OK;
}

int sptrsv_device_name(int device, char* buf, int len) {
    if (!buf || len <= 0) return fail(SPTRSV_E_INVALID_ARG, "bad buffer");
    hipDeviceProp_t p;
    SPT_HIP(hipGetDeviceProperties(&p, device));
    snprintf(buf, (size_t)len, "%s (%s, %d CUs)", p.name, p.gcnArchName, p.multiProcessorCount);
    return SPTRSV_OK;
}

int sptrsv_malloc(void** p, size_t bytes) {
    if (!p) return fail(SPTRSV_E_INVALID_ARG, "null pointer");
    SPT_HIP(hipMalloc(p, std::max<size_t>(bytes, 1)));
    return SPTRSV_OK;
}
int sptrsv_free(void* p) {
    if (p) SPT_HIP(hipFree(p));
    return SPTRSV_OK;
}
int sptrsv_memcpy_htod(void* dst, const void* src, size_t bytes) {
    if (bytes) SPT_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return SPTRSV_OK;
}
int sptrsv_memcpy_dtoh(void* dst, const void* src, size_t bytes) {
    if (bytes) SPT_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return SPTRSV_OK;
}
int sptrsv_memset(void* dst, int value, size_t bytes) {
    if (bytes) SPT_HIP(hipMemset(dst, value, bytes));
    return SPTRSV_OK;
}
int sptrsv_synchronize(void) {
    SPT_HIP(hipDeviceSynchronize());
    return SPTRSV_OK;
}
int sptrsv_copy_device(void* dst, const void* src, size_t bytes) {
    if (bytes % 16 || ((uintptr_t)dst | (uintptr_t)src) % 16)
        return fail(SPTRSV_E_INVALID_ARG, "copy needs 16-byte aligned pointers and size");
    const size_t n = bytes / 16;
    if (n == 0) return SPTRSV_OK;
    const unsigned g = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_copy16, dim3(g), dim3(256), 0, nullptr, static_cast<uint4*>(dst),
                       static_cast<const uint4*>(src), n);
    SPT_HIP(hipGetLastError());
    return SPTRSV_OK;
}

int sptrsv_timer_start(hipStream_t stream) {
    std::lock_guard<std::mutex> g(g_timer_mu);
    if (!g_t0) {
        SPT_HIP(hipEventCreate(&g_t0));
        SPT_HIP(hipEventCreate(&g_t1));
    }
    SPT_HIP(hipEventRecord(g_t0, stream));
    return SPTRSV_OK;
}

int sptrsv_timer_stop(hipStream_t stream, float* ms) {
    std::lock_guard<std::mutex> g(g_timer_mu);
    if (!g_t0 || !ms) return fail(SPTRSV_E_INVALID_ARG, "timer not started");
    SPT_HIP(hipEventRecord(g_t1, stream));
    SPT_HIP(hipEventSynchronize(g_t1));
    SPT_HIP(hipEventElapsedTime(ms, g_t0, g_t1));
    return SPTRSV_OK;
}

static uint4* g_flush_buf = nullptr;  // sptrsv_flush_cache's scratch

}  // extern "C"

namespace sptrsv {
// Library teardown, before the HIP runtime's own (this library is loaded
// after it, so it is unloaded first): captured graphs and capture streams of
// handles still alive, and the library's own events and scratch.  Device
// memory of live handles is left to the runtime.  Nothing here touches HIP
// unless such objects exist (a process that never used the GPU stays clear).
__attribute__((destructor)) static void interface_teardown() {
    std::lock_guard<std::mutex> g(g_live_mu);
    if (!g_live.empty() || g_t0 || g_flush_buf) (void)hipDeviceSynchronize();
    for (MatPriv* pv : g_live) {
        for (auto& gr : pv->graphs) (void)hipGraphExecDestroy(gr.second);
        pv->graphs.clear();
        if (pv->cap_stream) (void)hipStreamDestroy(pv->cap_stream);
        pv->cap_stream = nullptr;
    }
    if (g_t0) (void)hipEventDestroy(g_t0);
    if (g_t1) (void)hipEventDestroy(g_t1);
    g_t0 = g_t1 = nullptr;
    if (g_flush_buf) (void)hipFree(g_flush_buf);
    g_flush_buf = nullptr;
}
}  // namespace sptrsv

extern "C" {

static __global__ void k_flush(uint4* p, size_t count, unsigned salt) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (size_t)gridDim.x * blockDim.x)
        p[i] = make_uint4((unsigned)i, salt, (unsigned)i ^ salt, salt + 1);
}

int sptrsv_flush_cache(hipStream_t stream) {
    static unsigned salt = 0;
    const size_t bytes = 512ull << 20;  // twice the 256 MB Infinity Cache
    if (!g_flush_buf) SPT_HIP(hipMalloc(&g_flush_buf, bytes));
    hipLaunchKernelGGL(k_flush, dim3(4096), dim3(256), 0, stream, g_flush_buf, bytes / sizeof(uint4), ++salt);
    SPT_HIP(hipGetLastError());
    return SPTRSV_OK;
}

int sptrsv_measure_dep_latency(int rounds, float* one_way_ns) {
    if (rounds < 1 || !one_way_ns) return fail(SPTRSV_E_INVALID_ARG, "bad arguments");
    unsigned* flags = nullptr;
    long long* out = nullptr;
    SPT_HIP(hipMalloc(&flags, 64 * sizeof(unsigned)));
    SPT_HIP(hipMalloc(&out, 4 * sizeof(long long)));
    int dev = 0;
    SPT_HIP(hipGetDevice(&dev));
    int rate = 100000;
    (void)hipDeviceGetAttribute(&rate, hipDeviceAttributeWallClockRate, dev);
    std::vector<float> ns;
    int st = SPTRSV_OK;
    for (int partner = 1; partner < 8 && st == SPTRSV_OK; ++partner) {
        SPT_HIP(hipMemset(flags, 0, 64 * sizeof(unsigned)));
        SPT_HIP(hipMemset(out, 0, 4 * sizeof(long long)));
        hipLaunchKernelGGL(k_pingpong, dim3(16), dim3(64), 0, nullptr, flags, partner, rounds, out, 1 << 22);
        SPT_HIP(hipGetLastError());
        long long h[4];
        SPT_HIP(hipMemcpy(h, out, sizeof(h), hipMemcpyDeviceToHost));
        if (h[2]) st = fail(SPTRSV_E_WATCHDOG, "ping-pong wait exceeded its bound");
        else ns.push_back((float)(h[0] * (1e6 / rate) / (2.0 * rounds)));
    }
    (void)hipFree(flags);
    (void)hipFree(out);
    if (st != SPTRSV_OK) return st;
    std::sort(ns.begin(), ns.end());
    *one_way_ns = ns[ns.size() / 2];
    return SPTRSV_OK;
}

int sptrsv_bench_solve(sp_mat_t* mat, dfr_analysis_info_t* info, int precision,
                       const sptrsv_config_t* cfg, const void* b, void* x, int n, int k,
                       int refine_steps, int reps, int check_ones, sptrsv_bench_t* out) {
    if (!out || reps < 1) return fail(SPTRSV_E_INVALID_ARG, "bad bench arguments");
    // warm-up (allocates workspaces outside the timed loop)
    SPT_TRY(sptrsv_solve(mat, info, precision, cfg, b, x, n, k, refine_steps, nullptr));
    SPT_HIP(hipDeviceSynchronize());
    std::vector<hipEvent_t> ev(2 * reps);
    for (auto& e : ev) SPT_HIP(hipEventCreate(&e));
    int pw = amdsmiAPIRun("sptrsv_bench_solve", priv_of(mat)->device, 1000);
    int st = SPTRSV_OK;
    for (int r = 0; r < reps && st == SPTRSV_OK; ++r) {
        SPT_HIP(hipEventRecord(ev[2 * r], nullptr));
        st = sptrsv_solve(mat, info, precision, cfg, b, x, n, k, refine_steps, nullptr);
        SPT_HIP(hipEventRecord(ev[2 * r + 1], nullptr));
    }
    SPT_HIP(hipDeviceSynchronize());
    float power = pw == SPTRSV_OK ? amdsmiAPIEnd() : -1.0f;
    if (pw == SPTRSV_OK && amdsmiAPISamples() == 0) power = -1.0f;
    if (st != SPTRSV_OK) return st;
    // mean and stdev (BENCH_RUN_SOLVE keeps a running mean of squares, common.h:112-118)
    double sum = 0, sq = 0, mn = 1e30;
    for (int r = 0; r < reps; ++r) {
        float ms = 0;
        SPT_HIP(hipEventElapsedTime(&ms, ev[2 * r], ev[2 * r + 1]));
        sum += ms;
        sq += (double)ms * ms;
        mn = std::min<double>(mn, ms);
    }
    for (auto& e : ev) (void)hipEventDestroy(e);
    double mean = sum / reps;
    double var = sq / reps - mean * mean;
    out->mean_ms = (float)mean;
    out->stdev_ms = (float)sqrt(var > 0 ? var : 0);
    out->min_ms = (float)mn;
    out->power_mw = power;
    out->reps = reps;
    out->errors = -1;
    SPT_TRY(sptrsv_check(mat, nullptr));
    if (check_ones) {
        size_t cnt = (size_t)n * k;
        int errs = 0;
        if (precision == SPTRSV_PREC_F32) {
            std::vector<float> h(cnt);
            SPT_HIP(hipMemcpy(h.data(), x, cnt * sizeof(float), hipMemcpyDeviceToHost));
            for (float v : h) errs += (fabsf(1.0f - v) != 0.0f);
        } else {
            std::vector<double> h(cnt);
            SPT_HIP(hipMemcpy(h.data(), x, cnt * sizeof(double), hipMemcpyDeviceToHost));
            for (double v : h) errs += (fabs(1.0 - v) != 0.0);
        }
        out->errors = errs;
    }
    return SPTRSV_OK;
}

}  // extern "C"
