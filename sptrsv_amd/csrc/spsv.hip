// spsv.hip -- a generic triangular-solve handle over a device CSR matrix, in
// the shape of the vendor sparse libraries' SpSV call sequence (create,
// analysis, solve, destroy): fill mode, diagonal type and operation are
// arguments instead of properties of the upload.
//
// The handle is built on the device from the caller's CSR:
//  * only the chosen triangle is read (entries of the other one are
//    ignored);
//  * a unit diagonal ignores any stored diagonal entry; a non-unit diagonal
//    takes the row's first stored (i, i) entry, and a row without one is
//    SPTRSV_E_INVALID_CSR;
//  * a lower triangle is stored as is with the diagonal moved last; an upper
//    one is stored as the lower triangle of the reversed index order (row
//    n-1-i, columns n-1-j), which the solves undo on b and x;
//  * the transposed operation is the device transpose of that handle.
// The caller's arrays are not referenced after creation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "common.hpp"

namespace sptrsv {

int convert_values_to_f32(sp_mat_t* m);

namespace {

unsigned row_grid(long long count) {
    return (unsigned)std::max<long long>(1, std::min<long long>((count + 255) / 256, 16384));
}

// Stored-row lengths: kept off-diagonals + 1 (the diagonal) at the stored
// row (i, or n-1-i for an upper triangle); dpos[i] = the diagonal entry used
// (-1 for a unit diagonal); out[0] bit 1 = column outside [0, n), bit 2 = a
// missing diagonal; out[1] bit 1 = a kept column 64 or more rows
// away, 2 = one kept twice in a row; out[2] of the
// out[3] rows of every eighth workgroup have their nearest kept one within kNear,
// and out[4..5] is the sum of the distances to it of the out[8] rows that have
// one (in an upper triangle whose columns ascend it is the first one).
__global__ __launch_bounds__(256) void k_tri_count(const int* __restrict__ ia, const int* __restrict__ ja, int n,
                                                   int upper, int unit, int* __restrict__ len, int* __restrict__ dpos,
                                                   int* __restrict__ out) {
    int wide = 0, twice = 0, near = 0, rows = 0, waiting = 0;
    unsigned long long dist = 0;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x) {
        const int i = (int)t;
        int kept = 0, d = -1, flags = 0, nearest = 0;
        unsigned long long seen = 0;  // distances
        for (int p = ia[i]; p < ia[i + 1]; ++p) {
            const int j = ja[p];
            if (j < 0 || j >= n) flags |= 1;
            else if (j == i) { if (d < 0) d = p; }
            else if (upper ? j > i : j < i) {
                const int away = abs(i - j);
                nearest = kept ? min(nearest, away) : away;
                ++kept;
                if (away >= kWave) {
                    wide = 1;
                } else {
                    twice |= (seen >> away) & 1 ? 2 : 0;
                    seen |= 1ull << away;
                }
            }
        }
        if (!unit && d < 0) flags |= 2;
        if (flags) atomicOr(out, flags);
        len[upper ? n - 1 - i : i] = kept + 1;
        dpos[i] = unit ? -1 : d;
        near += kept > 0 && nearest <= kNear;
        dist += nearest;
        waiting += kept > 0;
        ++rows;
    }
    if ((wide | twice) && (out[1] | wide | twice) != out[1]) atomicOr(&out[1], wide | twice);
    if ((blockIdx.x & 7) == 0) {
        __shared__ int s_near, s_rows, s_waiting;
        __shared__ unsigned long long s_dist;
        if (threadIdx.x == 0) {
            s_near = s_rows = s_waiting = 0;
            s_dist = 0;
        }
        __syncthreads();
        if (near) atomicAdd(&s_near, near);
        atomicAdd(&s_rows, rows);
        if (waiting) atomicAdd(&s_waiting, waiting);
        atomicAdd(&s_dist, dist);
        __syncthreads();
        if (threadIdx.x == 0) {
            atomicAdd(&out[2], s_near);
            atomicAdd(&out[3], s_rows);
            atomicAdd(&out[8], s_waiting);
            atomicAdd(reinterpret_cast<unsigned long long*>(out + 4), s_dist);
        }
    }
}

// Writes stored row r of source row i: its kept entries in source order
// (columns mapped to n-1-j for an upper triangle), then the diagonal.
__global__ void k_tri_fill(const int* __restrict__ ia, const int* __restrict__ ja, const double* __restrict__ a,
                           int n, int upper, const int* __restrict__ dpos, const int* __restrict__ ia_s,
                           int* __restrict__ ja_s, double* __restrict__ a_s, int* __restrict__ perm) {
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x) {
        const int i = (int)t;
        const int r = upper ? n - 1 - i : i;
        int w = ia_s[r];
        for (int p = ia[i]; p < ia[i + 1]; ++p) {
            const int j = ja[p];
            if (j < 0 || j >= n || j == i || (upper ? j < i : j > i)) continue;
            ja_s[w] = upper ? n - 1 - j : j;
            a_s[w] = a[p];
            perm[w] = p;
            ++w;
        }
        ja_s[w] = r;
        a_s[w] = dpos[i] >= 0 ? a[dpos[i]] : 1.0;
        perm[w] = dpos[i];
    }
}

template <class T>
__global__ void k_scale(T* __restrict__ x, long long count, T alpha) {
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < count;
         t += (long long)gridDim.x * blockDim.x)
        x[t] *= alpha;
}

// The triangle of (ia, ja, a) as a handle of the non-transposed operation.
int build_triangle(int n, int nnz, const int* ia, const int* ja, const double* a, bool upper, bool unit,
                   sp_mat_t* m) {
    memset(m, 0, sizeof(*m));
    SPT_TRY(ensure_priv(m));
    m->nr = m->nc = n;
    priv_of(m)->reversed = upper;
    int st = SPTRSV_OK;
    auto chk = [&](hipError_t e, const char* what) {
        if (e != hipSuccess && st == SPTRSV_OK) st = hip_fail(e, what, __FILE__, __LINE__);
    };
    int *len = nullptr, *dpos = nullptr, *bad = nullptr, *ia_s = nullptr, *scratch = nullptr;
    Arena work;
    work.add(&len, (size_t)n + 1);
    work.add(&dpos, n);
    work.add(&bad, 9);
    work.add(&ia_s, (size_t)n + 1);
    work.add(&scratch, scan_scratch((long long)n + 1));
    void* tmp = nullptr;
    chk(work.get(&tmp), "hipMalloc triangle work");
    if (st == SPTRSV_OK) chk(hipMemset(len, 0, 4 * ((size_t)n + 1)), "clear lengths");
    if (st == SPTRSV_OK) chk(hipMemset(bad, 0, 36), "clear flag");
    if (st == SPTRSV_OK && n > 0) {
        hipLaunchKernelGGL(k_tri_count, dim3(row_grid(n)), dim3(256), 0, nullptr, ia, ja, n, upper ? 1 : 0,
                           unit ? 1 : 0, len, dpos, bad);
        chk(hipGetLastError(), "triangle count");
    }
    // row pointers, and the longest row, before what came out is looked at: one
    // wait for all
    if (st == SPTRSV_OK) st = exclusive_scan(len, ia_s, (long long)n + 1, nullptr, scratch);
    if (st == SPTRSV_OK && n > 0) st = longest_row(ia_s, n, bad + 6, nullptr);
    int h_out[9] = {};
    int total = 0;
    if (st == SPTRSV_OK) chk(hipMemcpy(h_out, bad, 36, hipMemcpyDeviceToHost), "read flag");
    const int h_bad = h_out[0];
    if (st == SPTRSV_OK && (h_bad & 1)) st = fail(SPTRSV_E_INVALID_CSR, "column index outside [0, n)");
    if (st == SPTRSV_OK && (h_bad & 2)) st = fail(SPTRSV_E_INVALID_CSR, "a row has no diagonal entry (non-unit diagonal)");
    if (st == SPTRSV_OK) chk(hipMemcpy(&total, ia_s + n, 4, hipMemcpyDeviceToHost), "read ia");
    m->nnz = total;
    const size_t ne = (size_t)std::max(total, 1);
    Arena keep;
    keep.add(&m->ia, (size_t)n + 1);
    keep.add(&m->ja, ne);
    keep.add(&m->a, ne);
    keep.add(&m->a32, ne);
    keep.add(&priv_of(m)->src_perm, ne);
    if (st == SPTRSV_OK) chk(keep.get(&priv_of(m)->block), "hipMalloc triangle");
    if (st == SPTRSV_OK)
        chk(hipMemcpyAsync(m->ia, ia_s, 4 * ((size_t)n + 1), hipMemcpyDeviceToDevice, nullptr), "copy ia");
    priv_of(m)->src_count = nnz;
    if (st == SPTRSV_OK && n > 0) {
        hipLaunchKernelGGL(k_tri_fill, dim3(row_grid(n)), dim3(256), 0, nullptr, ia, ja, a, n, upper ? 1 : 0, dpos,
                           m->ia, m->ja, m->a, priv_of(m)->src_perm);
        chk(hipGetLastError(), "triangle fill");
    }
    if (st == SPTRSV_OK) {
        RowShape shape;
        shape.longest = h_out[6];
        // of all rows, so scaled to the ones seen
        shape.long_rows = n > 0 ? (long long)h_out[7] * h_out[3] / n : 0;
        shape.wide = (h_out[1] & 1) != 0;
        shape.twice = (h_out[1] & 2) != 0;
        shape.near = h_out[2];
        shape.waiting = h_out[8];
        memcpy(&shape.dist, h_out + 4, sizeof(shape.dist));
        shape.install(priv_of(m), n, h_out[3]);
    }
    if (st == SPTRSV_OK) st = convert_values_to_f32(m);
    if (st == SPTRSV_OK) chk(hipDeviceSynchronize(), "triangle sync");
    if (tmp) (void)hipFree(tmp);
    if (st != SPTRSV_OK) free_mat(m);
    return st;
}

}  // namespace
}  // namespace sptrsv

using namespace sptrsv;

struct sptrsv_spsv {
    sp_mat_t mat{};
    dfr_analysis_info_t info{};
    bool analysed = false;
};

extern "C" {

int sptrsv_spsv_create(sptrsv_spsv_t** out, int n, int nnz, const int* d_ia, const int* d_ja, const double* d_a,
                       int fill, int diag, int op) {
    if (!out) return fail(SPTRSV_E_INVALID_ARG, "null handle pointer");
    *out = nullptr;
    if (n < 0 || nnz < 0 || (n > 0 && (!d_ia || (nnz > 0 && (!d_ja || !d_a)))))
        return fail(SPTRSV_E_INVALID_ARG, "bad CSR arguments");
    if ((fill != SPTRSV_FILL_LOWER && fill != SPTRSV_FILL_UPPER) ||
        (diag != SPTRSV_DIAG_NON_UNIT && diag != SPTRSV_DIAG_UNIT) ||
        (op != SPTRSV_OP_NONE && op != SPTRSV_OP_TRANSPOSE))
        return fail(SPTRSV_E_INVALID_ARG, "unknown fill mode, diagonal type or operation");
    auto* h = new sptrsv_spsv();
    sp_mat_t tri{};
    int st = build_triangle(n, nnz, d_ia, d_ja, d_a, fill == SPTRSV_FILL_UPPER, diag == SPTRSV_DIAG_UNIT, &tri);
    if (st == SPTRSV_OK && op == SPTRSV_OP_TRANSPOSE) {
        st = sptrsv_transpose(&tri, &h->mat);
        free_mat(&tri);
    } else if (st == SPTRSV_OK) {
        h->mat = tri;
    }
    if (st != SPTRSV_OK) {
        delete h;
        return st;
    }
    *out = h;
    return SPTRSV_OK;
}

int sptrsv_spsv_analysis(sptrsv_spsv_t* h, int precision, int k, int tune) {
    if (!h) return fail(SPTRSV_E_INVALID_ARG, "null handle");
    if (h->analysed) free_device_analysis(nullptr, &h->info);
    h->analysed = false;
    dfr_analysis_info_t* p = &h->info;
    // often for one solve, and solved with the shape an ALL analysis has by
    // default, which needs no plan (with one, random n = 3000 took 7 % longer)
    SPT_TRY(level_analysis(&p, &h->mat, ALL, false));
    h->analysed = true;
    if (tune && h->mat.nr > 0) {
        sptrsv_config_t best{};
        float ms = 0;
        SPT_TRY(sptrsv_autotune(&h->mat, &h->info, precision, std::max(k, 1), 3, &best, &ms));
    }
    return SPTRSV_OK;
}

int sptrsv_spsv_solve(sptrsv_spsv_t* h, int precision, double alpha, const void* b, void* x, int k,
                      hipStream_t stream) {
    if (!h) return fail(SPTRSV_E_INVALID_ARG, "null handle");
    SPT_TRY(sptrsv_solve(&h->mat, h->analysed ? &h->info : nullptr, precision, nullptr, b, x, h->mat.nr, k, 1,
                         stream));
    if (alpha != 1.0 && h->mat.nr > 0) {
        const long long count = (long long)h->mat.nr * k;
        if (precision == SPTRSV_PREC_F32)
            hipLaunchKernelGGL(k_scale<float>, dim3(row_grid(count)), dim3(256), 0, stream, static_cast<float*>(x),
                               count, (float)alpha);
        else
            hipLaunchKernelGGL(k_scale<double>, dim3(row_grid(count)), dim3(256), 0, stream, static_cast<double*>(x),
                               count, alpha);
        SPT_HIP(hipGetLastError());
    }
    return SPTRSV_OK;
}

sp_mat_t* sptrsv_spsv_matrix(sptrsv_spsv_t* h) { return h ? &h->mat : nullptr; }

void sptrsv_spsv_destroy(sptrsv_spsv_t* h) {
    if (!h) return;
    free_device_analysis(&h->mat, h->analysed ? &h->info : nullptr);
    delete h;
}

}  // extern "C"
