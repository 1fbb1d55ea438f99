// level_walk.hip -- the level walk (variant 4): one workgroup solves an
// analysed matrix level by level, exchanging results through LDS.
//
// For matrices with few rows per level a dependency hop through memory is
// what every other walk waits for: about 365 ns from one XCD to another and
// 210 ns inside one even when idle, and two to three times that with a
// thousand polling waves.  Inside one workgroup a level costs a barrier (20 to
// 25 ns) and an LDS gather: there are no flags, no polls and nothing to clear
// before a solve.  The price is that one CU streams the whole matrix, so the
// walk is taken while a level's share of the matrix is small (see
// level_walk_fits).
//
// What bounds it then is the instructions of a step: a wave issues one every
// four cycles, so the plan holds everything in the form the walk uses it, and
// a step of a wave is about 40 instructions (addresses computed in the kernel
// made it 450, and the walk five times slower).
//
// Plan (built on the device for one matrix and analysis, with the analysis where
// the walk is a default and else on the first solve that names it; its
// records are written before every walk, see k_lw_fill): slices
// of 64 / L rows of one level and one row-length group, L lanes per row so
// that a lane has at most kLwU entries.  A step is NW slices of a level, one
// per wave, closed by a barrier.  Slices have a fixed size: kLwU records per
// lane (LDS address of the dependency's word, value) and one row record (index
// of the row's own word, byte offset of the row in b and x, 1 / diagonal),
// lane-interleaved, so every load of a step is one fully coalesced instruction
// with no address arithmetic.  Lanes without an entry read a word that is
// always 0; lanes without a row write to a spare word, and their offset in b
// and x is beyond the buffers, whose range check drops the access; a wave
// without a slice in a step reads beyond the buffers likewise.
//
// The words of at least the last 8192 positions are in an LDS ring (128 KB for
// 8-byte words).  An entry that reaches further back (far) has a record of its
// own and reads the words in memory (x itself, or for the fused mixed pass a
// copy of the words), written at least 4096 positions and a full barrier before
// (see the end of a step).  Entries for which a lane has no record left are in an
// overflow list of their slice.
//
// Measured (default shape of csr_L_solve_order / _multirow before -> now): 2D
// grid factor of 64^2 (127 levels) 120 -> 27 us, of 250^2 516 -> 130 us, 3D grid
// 15^3 54 -> 21 us, random n = 2000 95 -> 31 us: 0.15 to 0.2 us a level while a
// step is one or two slices, 0.55 us with eight (the CU then takes in about 65
// GB/s), and 5 us for the launch that writes the records.
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "syncfree.hpp"

namespace sptrsv {

constexpr int kLwU = 4;                    // records per lane and slice
constexpr int kLwRing = 16384;             // words in LDS
constexpr int kLwEpoch = kLwRing / 4;
constexpr unsigned kLwNone = 0xffffffffu;  // byte offset out of every buffer's range
// First position whose word is still in the ring for a slice at position pos:
// two epochs before its own (the ring holds four, a step at most 512 rows).
__host__ __device__ constexpr int lw_near(int pos) { return (pos / kLwEpoch - 2) * kLwEpoch; }
// LDS words: one spare word per lane (word 0 is also what a record of zeros,
// read beyond a buffer, names), a word that stays 0, the ring.
constexpr int kLwZero = kWave, kLwRing0 = kWave + 1, kLwWords = kLwRing0 + kLwRing;
// First word of a row record: word index, log2(L), overflow flag.
constexpr unsigned kLwIndexBits = 18, kLwOverflow = 1u << 21;
static_assert(kLwWords <= (1 << kLwIndexBits), "word index field");
// Slots (plan): position + 1 of a near dependency, or row + 1 of a far one with
// bit 31; 0: none.
constexpr unsigned kLwFar = 0x80000000u;
// Step table: first slice << 4 | slices; bit 31: ends with a full barrier.
constexpr unsigned kLwStepFlush = 0x80000000u;
constexpr int kLwMaxSlices = 1 << 19;  // keeps every buffer under 2 GB

// ---- plan kernels ---------------------------------------------------------------

struct LwShape {
    int nw;       // waves of the workgroup
    int lg_big;   // log2(L) of rows with more than 16 off-diagonals
};

// Groups of a level's rows, consecutive in iorder: row-length classes {0, 1,
// 2} (1 to 4 off-diagonals), 3 (to 8), 4 (to 16), 5 and 6 (diagonal only).
__device__ __forceinline__ int lw_group_lg(int group, const LwShape& s) {
    return group == 1 ? 1 : group == 2 ? 2 : group == 3 ? s.lg_big : 0;
}
__device__ __forceinline__ void lw_group_range(const int* __restrict__ bucket_off, int lev, int g, int* lo, int* hi) {
    *lo = bucket_off[7 * lev + (g == 0 ? 0 : g + 2)];
    *hi = bucket_off[7 * lev + g + 3];
}

// Slices and steps of every level (per[l] and per[nlevs + 1 + l]).
__global__ void k_lw_count(const int* __restrict__ bucket_off, int nlevs, LwShape sh, int* __restrict__ slices,
                           int* __restrict__ steps, int* __restrict__ flags) {
    if (blockIdx.x == 0 && threadIdx.x < 3) flags[threadIdx.x] = 0;
    for (int l = blockIdx.x * blockDim.x + threadIdx.x; l <= nlevs; l += gridDim.x * blockDim.x) {
        int sl = 0;
        if (l < nlevs)
            for (int g = 0; g < 5; ++g) {
                int lo, hi;
                lw_group_range(bucket_off, l, g, &lo, &hi);
                const int rps = kWave >> lw_group_lg(g, sh);
                sl += (hi - lo + rps - 1) / rps;
            }
        slices[l] = sl;
        steps[l] = (sl + sh.nw - 1) / sh.nw;
    }
}

// Slices (x = first position, y = rows | log2(L) << 8 | flush << 16) and the
// step table, whose entries from the last step on to steps_all are empty.
__global__ void k_lw_slices(const int* __restrict__ bucket_off, int nlevs, LwShape sh, const int* __restrict__ slice_off,
                            const int* __restrict__ step_off, int steps_all, int2* __restrict__ slice,
                            unsigned* __restrict__ step) {
    const int t0 = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
    for (int t = step_off[nlevs] + t0; t < steps_all; t += stride) step[t] = 0;
    for (int l = t0; l < nlevs; l += stride) {
        const int begin = slice_off[l], end = slice_off[l + 1], last = bucket_off[7 * (l + 1)];
        int s = begin;
        for (int g = 0; g < 5; ++g) {
            int lo, hi;
            lw_group_range(bucket_off, l, g, &lo, &hi);
            const int lg = lw_group_lg(g, sh), rps = kWave >> lg;
            for (int p = lo; p < hi; p += rps) slice[s++] = make_int2(p, min(rps, hi - p) | (lg << 8));
        }
        int t = step_off[l];
        for (s = begin; s < end; s += sh.nw, ++t) {
            const int c = min(sh.nw, end - s);
            step[t] = ((unsigned)s << 4) | (unsigned)c;
            // a step whose positions reach a new epoch ends with a full barrier
            const int p1 = s + c < end ? slice[s + c].x : last;
            if (slice[s].x / kLwEpoch != p1 / kLwEpoch) step[t] |= kLwStepFlush;
        }
    }
}

// Slots of every slice, a wave each: lane e of a row takes its entries e, e +
// L, ... in storage order into its kLwU near slots and its far slot, and the
// rest into the slice's overflow list (a count of slots per lane, then that
// many for every lane).  flags: [0] bits 1: a column is not at an earlier level
// (the analysis is another matrix's), 2: no room for an overflow list; [1]
// overflow slots used; [2] far entries.
__global__ void k_lw_slots(const int* __restrict__ ia, const int* __restrict__ ja, const int* __restrict__ iorder,
                           const int* __restrict__ inv, const int* __restrict__ level, bool by_position,
                           const int2* __restrict__ slice, int n_slices, unsigned* __restrict__ col, int* __restrict__ from, unsigned* __restrict__ fcol,
                           int* __restrict__ ffrom, int* __restrict__ over, unsigned* __restrict__ ocol,
                           int* __restrict__ ofrom, int over_cap, int* __restrict__ diag_from, int* __restrict__ order,
                           int* __restrict__ flags) {
    const int lane = threadIdx.x & (kWave - 1);
    const int waves = (gridDim.x * blockDim.x) / kWave;
    int bad = 0, far_all = 0;
    for (int s = (blockIdx.x * blockDim.x + threadIdx.x) / kWave; s < n_slices; s += waves) {
        const int2 d = slice[s];
        const int rows = d.y & 255, lg = (d.y >> 8) & 255, rl = lane >> lg, e = lane & ((1 << lg) - 1);
        int q0 = 0, q1 = 0, lev = 0;
        const int lo = lw_near(d.x);
        if (rl < rows) {
            const int r = iorder[d.x + rl];
            q1 = ia[r + 1] - 1;
            q0 = ia[r] + e;
            lev = level[r];
            if (e == 0) {
                diag_from[d.x + rl] = q1;
                order[d.x + rl] = r;
            }
        }
        unsigned c[kLwU] = {}, fc = 0;
        int f[kLwU], ff = -1, nn = 0, nf = 0, no = 0;
        for (int u = 0; u < kLwU; ++u) f[u] = -1;
        for (int q = q0; q < q1; q += 1 << lg) {
            const int j = ja[q], p = inv[j];
            if (level[j] >= lev) bad = 1;
            if (p >= lo && nn < kLwU) {
#pragma unroll
                for (int u = 0; u < kLwU; ++u)
                    if (u == nn) {
                        c[u] = (unsigned)p + 1u;
                        f[u] = q;
                    }
                ++nn;
            } else if (p < lo && nf == 0) {
                fc = (unsigned)((by_position ? p : j) + 1) | kLwFar;
                ff = q;
                ++nf;
            } else {
                ++no;
            }
            far_all += p < lo;
        }
        int most = no;
        for (int o = 1; o < kWave; o <<= 1) most = max(most, __shfl_xor(most, o));
        int at = -1;
        if (most) {
            if (lane == 0) at = atomicAdd(&flags[1], 1 + most);
            at = __shfl(at, 0);
            if (at < 0 || at + 1 + most > over_cap) {
                bad |= 2;
                at = -1;
            }
        }
        if (lane == 0) over[s] = at;
        if (at >= 0) {
            // unit at: the count in its first slot; then a unit of 64 slots per entry
            ocol[(size_t)at * kWave + lane] = lane == 0 ? (unsigned)most : 0u;
            ofrom[(size_t)at * kWave + lane] = -1;
            int kn = 0, kf = 0, k = 0;
            for (int q = q0; q < q1; q += 1 << lg) {
                const int j = ja[q], p = inv[j];
                if (p >= lo && kn < kLwU) {
                    ++kn;
                } else if (p < lo && kf == 0) {
                    ++kf;
                } else {
                    ocol[(size_t)(at + 1 + k) * kWave + lane] = p < lo ? (unsigned)((by_position ? p : j) + 1) | kLwFar : (unsigned)p + 1u;
                    ofrom[(size_t)(at + 1 + k) * kWave + lane] = q;
                    ++k;
                }
            }
            for (; k < most; ++k) {
                ocol[(size_t)(at + 1 + k) * kWave + lane] = 0;
                ofrom[(size_t)(at + 1 + k) * kWave + lane] = -1;
            }
        }
#pragma unroll
        for (int u = 0; u < kLwU; ++u) {
            col[((size_t)s * kLwU + u) * kWave + lane] = c[u];
            from[((size_t)s * kLwU + u) * kWave + lane] = f[u];
        }
        fcol[(size_t)s * kWave + lane] = fc;
        ffrom[(size_t)s * kWave + lane] = ff;
    }
    for (int o = 1; o < kWave; o <<= 1) {
        bad |= __shfl_xor(bad, o);
        far_all += __shfl_xor(far_all, o);
    }
    if (lane == 0 && bad) atomicOr(&flags[0], bad);
    if (lane == 0 && far_all) atomicAdd(&flags[2], far_all);
}

// Before every walk, the records in the form it uses them, from the values the
// matrix holds then: sp_mat_t::a and a32 may be written in place between solves.
// The launch costs 5 us (2D grid factor 64^2, 22.1 -> 27.5 us) and 60 MB of
// traffic over the whole device at 707^2, where it replaces a rewrite of the
// records at every value update (two updates and two solves 1803 -> 1693 us).
template <class T>
struct LwFill {
    const int2* slice;
    int n_slices;
    const unsigned *col, *fcol, *ocol;
    const int *from, *ffrom, *ofrom;
    long long n_over_slots;
    const int *over, *order, *diag_from;
    const T* a;
    unsigned *rec, *frec, *orec, *rowrec;  // frec null: no far entries
    float* piv32;
    const T* b;  // b into position order (bp null: the walk reads it in place)
    T* bp;
    int n;
};

// Record of a slot: the value, then the LDS byte address of a near dependency's
// word, or the byte offset of a far one's in memory (kLwNone: none).
template <class T>
__device__ __forceinline__ void lw_record(unsigned c, int q, bool far, const T* __restrict__ a, unsigned* __restrict__ rec,
                                          size_t i) {
    constexpr int W = 1 + sizeof(T) / 4;
    const T v = c && q >= 0 ? a[q] : T(0);
    unsigned w[W - 1];
    __builtin_memcpy(w, &v, sizeof(T));
    const unsigned p = (c & ~kLwFar) - 1u;
#pragma unroll
    for (int j = 0; j + 1 < W; ++j) rec[i * W + j] = w[j];
    rec[i * W + W - 1] = far ? (c ? p * (unsigned)sizeof(T) : kLwNone)
                             : (c ? kLwRing0 + (p & (kLwRing - 1)) : (unsigned)kLwZero) * (unsigned)sizeof(T);
}

// Slot records and row records, a wave per slice; overflow records; b.  Row
// record of every lane: word index and flags, the complement of the row's byte
// offset in b and x (of its position's where b passes through position order),
// then the reciprocal of the diagonal (FP64, FP32) or the diagonal, with piv32
// its reciprocal in FP32 (mixed).
// b goes into position order, and x out of it, for matrices of more than
// kLwInPlace rows: the rows of a level are scattered over b and x, and a gather
// of 8 bytes costs the one CU that walks a whole line.
template <class T, bool MIXED>
__global__ void k_lw_fill(LwFill<T> F) {
    constexpr int W = 2 + sizeof(T) / 4;
    const int lane = threadIdx.x & (kWave - 1);
    const long long t0 = (long long)blockIdx.x * blockDim.x + threadIdx.x, stride = (long long)gridDim.x * blockDim.x;
    for (long long s = t0 / kWave; s < F.n_slices; s += stride / kWave) {
        const int2 d = F.slice[s];
        const int rows = d.y & 255, lg = (d.y >> 8) & 255, rl = lane >> lg;
#pragma unroll
        for (int u = 0; u < kLwU; ++u) {
            const size_t i = ((size_t)s * kLwU + u) * kWave + lane;
            lw_record(F.col[i], F.from[i], false, F.a, F.rec, i);
        }
        const size_t i = (size_t)s * kWave + lane;
        if (F.frec) lw_record(F.fcol[i], F.ffrom[i], true, F.a, F.frec, i);
        const unsigned flags = ((unsigned)lg << kLwIndexBits) | (F.over[s] >= 0 ? kLwOverflow : 0u);
        unsigned r[4] = {(unsigned)lane | flags, ~kLwNone, 0u, 0u};
        float p32 = 0.0f;
        if (rl < rows && (lane & ((1 << lg) - 1)) == 0) {
            const int p = d.x + rl;
            const T dg = F.a[F.diag_from[p]];
            T v = MIXED ? dg : T(1) / dg;
            if (MIXED) p32 = 1.0f / (float)dg;
            r[0] = (unsigned)(kLwRing0 + (p & (kLwRing - 1))) | flags;
            r[1] = ~((unsigned)(F.bp ? p : F.order[p]) * (unsigned)sizeof(T));
            __builtin_memcpy(r + 2, &v, sizeof(T));
        }
#pragma unroll
        for (int j = 0; j < W; ++j) F.rowrec[i * W + j] = r[j];
        if (MIXED) F.piv32[i] = p32;
    }
    for (long long i = t0; i < F.n_over_slots; i += stride) lw_record(F.ocol[i], F.ofrom[i], false, F.a, F.orec, i);
    if (F.bp)
        for (long long p = t0; p < F.n; p += stride) F.bp[p] = F.b[F.order[p]];
}

template <class T>
__global__ void k_lw_scatter(const T* __restrict__ src, const int* __restrict__ order, int n, T* __restrict__ dst) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x)
        __builtin_nontemporal_store(src[p], &dst[order[p]]);
}
constexpr int kLwInPlace = 16384;

// ---- the walk -----------------------------------------------------------------------

struct LwArgs {
    int nsteps;
    const unsigned* step;  // step table, whole blocks of 64 with 64 empty steps at the end
    const void* rec;       // slot records
    const void* frec;      // far slot records
    const void* rows;      // row records
    const float* piv32;    // mixed: 1 / diagonal in FP32, per lane
    const int* over;       // first overflow unit of a slice, -1 for none
    const void* orec;      // overflow records
    const unsigned* ocol;  // and slots
    const void* b;
    void* x;
    void* pub;             // mixed: words by row, for far entries
    unsigned n, n_steps_all, n_slices;
};

using Rsrc = __amdgpu_buffer_rsrc_t;
using U32x2 = unsigned __attribute__((ext_vector_type(2)));
using U32x3 = unsigned __attribute__((ext_vector_type(3)));
using U32x4 = unsigned __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Rsrc lw_rsrc(const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(unsigned)bytes, 0x00027000);
}
// W words at byte offsets off (per lane) + soff (of the wave).  AUX = 16 (sc1)
// reads past the CU's L1.
template <int W, int AUX = 0>
__device__ __forceinline__ auto lw_load(Rsrc r, unsigned off, unsigned soff = 0) {
    if constexpr (W == 1) return (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, (int)soff, AUX);
    else if constexpr (W == 2)
        return __builtin_bit_cast(U32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, (int)soff, AUX));
    else if constexpr (W == 3)
        return __builtin_bit_cast(U32x3, __builtin_amdgcn_raw_buffer_load_b96(r, (int)off, (int)soff, AUX));
    else return __builtin_bit_cast(U32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, AUX));
}
__device__ __forceinline__ void lw_store(Rsrc r, unsigned off, U32x2 v) {
    __builtin_amdgcn_raw_buffer_store_b64(v, r, (int)off, 0, 0);
}
__device__ __forceinline__ void lw_store(Rsrc r, unsigned off, unsigned v) {
    __builtin_amdgcn_raw_buffer_store_b32(v, r, (int)off, 0, 0);
}
__device__ __forceinline__ double lw_f64(unsigned lo, unsigned hi) {
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ double lw_f64(U32x2 v) { return lw_f64(v.x, v.y); }
__device__ __forceinline__ U32x2 lw_words(double v) { return __builtin_bit_cast(U32x2, v); }
__device__ __forceinline__ uint64_t lw_word(U32x2 v) { return ((uint64_t)v.y << 32) | v.x; }
__device__ __forceinline__ uint32_t lw_word(unsigned v) { return v; }

// What each policy reads and writes.  Results need no canonical NaN here:
// nothing takes a word for a flag.
template <class P>
struct LwOps;
template <>
struct LwOps<PolF64> {
    static constexpr int V = 2;  // 32-bit words of a value
    using Rec = U32x3;
    using Num = U32x2;
    using Row = U32x4;
    __device__ static unsigned at(const Rec& r) { return r.z; }
    __device__ static PolF64::Val val(const Rec& r) { return {lw_f64(r.x, r.y)}; }
    __device__ static PolF64::Acc seed(Num b) { return {lw_f64(b)}; }
    __device__ static uint64_t finish(const Row& row, float, const PolF64::Acc& t, Num* x) {
        *x = lw_words(t.s * lw_f64(row.z, row.w));
        return lw_word(*x);
    }
};
template <>
struct LwOps<PolMixed> {
    static constexpr int V = 2;
    using Rec = U32x3;
    using Num = U32x2;
    using Row = U32x4;
    __device__ static unsigned at(const Rec& r) { return r.z; }
    // the FP32 values are the FP64 ones rounded, as in the matrix's own copy
    __device__ static PolMixed::Val val(const Rec& r) { return {(float)lw_f64(r.x, r.y), lw_f64(r.x, r.y)}; }
    __device__ static PolMixed::Acc seed(Num b) { return {(float)lw_f64(b), 0.0f, lw_f64(b)}; }
    __device__ static uint64_t finish(const Row& row, float piv32, const PolMixed::Acc& t, Num* x) {
        PolMixed::Out o{};
        const uint64_t w = PolMixed::finish(SolveArgs{}, {piv32, lw_f64(row.z, row.w)}, t, o);
        *x = lw_words(o.x);
        return w;
    }
};
template <>
struct LwOps<PolF32> {
    static constexpr int V = 1;
    using Rec = U32x2;
    using Num = unsigned;
    using Row = U32x3;
    __device__ static unsigned at(const Rec& r) { return r.y; }
    __device__ static PolF32::Val val(const Rec& r) { return {__uint_as_float(r.x)}; }
    __device__ static PolF32::Acc seed(Num b) { return {__uint_as_float(b)}; }
    __device__ static uint32_t finish(const Row& row, float, const PolF32::Acc& t, Num* x) {
        *x = __float_as_uint(t.s * __uint_as_float(row.z));
        return *x;
    }
};

// Loads come back in the order they were issued, so a wave that waits for one
// has waited for all before it: what step s folds is loaded D steps ahead, and
// what the addresses of those loads need (row and far records) 2 D steps.
template <class P, int WG, int D, bool FAR>
__global__ __launch_bounds__(WG) void k_level_walk(LwArgs A) {
    using O = LwOps<P>;
    using word = typename P::word;
    using Rec = typename O::Rec;
    using Num = typename O::Num;
    using Row = typename O::Row;
    constexpr int RW = 2 + O::V;  // words of a row record
    constexpr int DD = 2 * D, RB = sizeof(word) + 4;  // bytes of a slot record
    constexpr bool MIXED = std::is_same<P, PolMixed>::value;
    __shared__ word lds[kLwWords];
    const int lane = threadIdx.x & (kWave - 1);
    const unsigned wv = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (threadIdx.x == 0) lds[kLwZero] = 0;
    __syncthreads();
    const size_t slots = (size_t)A.n_slices * kWave;
    const Rsrc r_step = lw_rsrc(A.step, (size_t)A.n_steps_all * 4);
    const Rsrc r_rec = lw_rsrc(A.rec, slots * kLwU * RB);
    const Rsrc r_frec = lw_rsrc(FAR ? A.frec : nullptr, FAR ? slots * RB : 0);
    const Rsrc r_rows = lw_rsrc(A.rows, slots * (4 * RW));
    const Rsrc r_piv = lw_rsrc(MIXED ? A.piv32 : nullptr, MIXED ? slots * 4 : 0);
    const Rsrc r_b = lw_rsrc(A.b, (size_t)A.n * (4 * O::V));
    const Rsrc r_x = lw_rsrc(A.x, (size_t)A.n * (4 * O::V));
    // words of far dependencies: x itself, or the mixed pass's copy
    const Rsrc r_pub = FAR && MIXED ? lw_rsrc(A.pub, (size_t)A.n * sizeof(word)) : r_x;
    const unsigned v_rec = (unsigned)(lane * RB), v_row = (unsigned)(lane * (4 * RW)), v_piv = (unsigned)lane * 4u;

    unsigned tcur = 0, tnext;  // lane i: table entry of step (block * 64 + i)
    unsigned ent[DD];          // table entry of the step in each stage (wave-uniform)
    Row row[DD];
    Rec frec[DD];
    Rec rec[D][kLwU];
    Num bv[D], fword[D];
    float piv[D];

    auto load_block = [&](int blk) { return lw_load<1>(r_step, (unsigned)lane * 4u, (unsigned)blk * 256u); };
    // this wave's slice in a step, and what takes the lanes' offsets beyond the
    // buffers when it has none
    auto slice_of = [&](unsigned t) { return ((t & ~kLwStepFlush) >> 4) + wv; };
    auto beyond = [&](unsigned t) { return wv < (t & 15u) ? 0u : 0x80000000u; };
    auto first_loads = [&](int j, int q) {
        ent[j] = (unsigned)__builtin_amdgcn_readlane((int)tcur, q & 63);
        const unsigned sl = beyond(ent[j]) ? 0u : slice_of(ent[j]), off = beyond(ent[j]);
        row[j] = lw_load<RW>(r_rows, v_row + off, sl * (unsigned)(kWave * 4 * RW));
        if constexpr (FAR) frec[j] = lw_load<O::V + 1>(r_frec, v_rec + off, sl * (unsigned)(kWave * RB));
    };
    auto second_loads = [&](int j2, int j) {
        const unsigned off = beyond(ent[j2]), sl = off ? 0u : slice_of(ent[j2]);
        const unsigned v = v_rec + off, so = sl * (unsigned)(kLwU * kWave * RB);
#pragma unroll
        for (int u = 0; u < kLwU; ++u) rec[j][u] = lw_load<O::V + 1>(r_rec, v + u * (kWave * RB), so);
        bv[j] = lw_load<O::V>(r_b, ~row[j2].y);
        piv[j] = 0.0f;
        if constexpr (MIXED) piv[j] = __uint_as_float(lw_load<1>(r_piv, v_piv + off, sl * (kWave * 4u)));
        if constexpr (FAR) fword[j] = lw_load<O::V, 16>(r_pub, O::at(frec[j2]));
    };
    auto lds_word = [&](unsigned byte) -> word { return *reinterpret_cast<word*>(reinterpret_cast<char*>(lds) + byte); };
    auto step = [&](int j2, int j) {
        // a lane's entries after the first in a sum of their own (rounding error
        // against a row per wave: 0.9, and 1.07 with all in one)
        typename P::Acc acc = O::seed(bv[j]), rest = P::zero();  // 0 in lanes without a row
        word w[kLwU];
#pragma unroll
        for (int u = 0; u < kLwU; ++u) w[u] = lds_word(O::at(rec[j][u]));
#pragma unroll
        for (int u = 0; u < kLwU; ++u) P::fold(u == 0 ? acc : rest, O::val(rec[j][u]), w[u]);
        if constexpr (FAR) P::fold(rest, O::val(frec[j2]), lw_word(fword[j]));
        const unsigned z = (unsigned)__builtin_amdgcn_readfirstlane((int)row[j2].x);
        if (z & kLwOverflow) {  // entries beyond the lane's records
            const int at = A.over[slice_of(ent[j2])];
            const int count = (int)A.ocol[(size_t)at * kWave];
#pragma unroll 1
            for (int k = 1; k <= count; ++k) {
                const size_t i = (size_t)(at + k) * kWave + lane;
                const unsigned c = A.ocol[i];
                Rec r;
                __builtin_memcpy(&r, static_cast<const char*>(A.orec) + i * RB, RB);
                word g = 0;
                if (c & kLwFar)
                    g = lw_word(lw_load<O::V, 16>(r_pub, ((c & ~kLwFar) - 1u) * (unsigned)sizeof(word)));
                else if (c)
                    g = lds[kLwRing0 + ((c - 1u) & (kLwRing - 1))];
                P::fold(rest, O::val(r), g);
            }
        }
        acc = P::add(acc, rest);
        const int lg = (int)(z >> kLwIndexBits) & 7;
        if (lg) acc = group_reduce<P, 1>(acc, 1 << lg);
        Num xv;
        const word res = O::finish(row[j2], piv[j], acc, &xv);
        lds[row[j2].x & ((1u << kLwIndexBits) - 1u)] = res;
        lw_store(r_x, ~row[j2].y, xv);
        if constexpr (FAR && MIXED) lw_store(r_pub, ~row[j2].y, __builtin_bit_cast(Num, res));
        if (FAR && (ent[j2] & kLwStepFlush)) {
            // A step that enters a new epoch: the words of the epoch before the one
            // just left are in memory for every wave.  The barrier alone does not
            // wait for stores; each wave has, in the steps of a whole epoch (at
            // least eight, of at most 512 rows), waited for loads it issued after
            // them, and vector memory operations of a wave are counted in order.
            // A far entry is more than an epoch back when its load goes out, D
            // steps ahead (lw_near).
            __syncthreads();
        } else {
            // results reach the other waves through LDS: wait for LDS only
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        }
    };

    tcur = load_block(0);
    tnext = load_block(1);
#pragma unroll
    for (int j = 0; j < DD; ++j) first_loads(j, j);
#pragma unroll
    for (int j = 0; j < D; ++j) second_loads(j, j);
    static_assert(64 % DD == 0, "a block of the step table is read by whole rounds");
    for (int q = DD; q - DD < A.nsteps; q += DD) {
        if ((q & 63) == 0) {
            tcur = tnext;
            tnext = load_block((q >> 6) + 1);
        }
#pragma unroll
        for (int j = 0; j < DD; ++j) {
            step(j, j % D);  // step q - DD + j; steps past the last one are empty
            second_loads((j + D) % DD, j % D);
            first_loads(j, q + j);
        }
    }
}

// ---- host ------------------------------------------------------------------------------

// A level's share of the matrix up to which one CU streaming it all, its records
// written before, beats the walks that need no plan (and is worth one: 50 to 90
// us of an analysis of 4000 rows).  Level walk against the best of the others,
// us, FP64 (mixed):
//  * rows of at most kLwU off-diagonals, a lane each: 131 / 248 (189 / 265) at
//    8.3 KB (2D grid 250^2), 354 / 397 (418 / 424) at 13.3 KB, 454 / 497 (529 /
//    533) at 16.6, 624 / 603 (730 / 649) at 19.9 (600^2), 820 / 722 at 23.5;
//  * rows of up to kLongRow, spread over lanes with room left over: 31 / 45 (42
//    / 49) at 3.4 KB (random n = 2000), 41 / 54 (54 / 59) at 5.9 KB, 62 / 59
//    (71 / 64) at 8.1;
//  * longer ones take a slice each: 50 / 52 (64 / 58) at 4.8 KB (power-law n =
//    2000), 73 / 58 at 6.8; never.
constexpr double kLwLevelBytes = 6.0 * 1024.0, kLwShortLevelBytes = 16.0 * 1024.0;
constexpr long long kLwMaxEntries = 1ll << 27;  // buffer descriptors address 4 GB
// Share of far entries above which the walk is not taken (their loads wait).
constexpr double kLwFarShare = 0.01;
// Device memory of a plan: bytes per slice (slots, records, rows), and what it
// may take per entry of the matrix and in any case.
constexpr double kLwSliceBytes = 64.0 * (kLwU * 20 + 20 + 16), kLwPlanShare = 96.0, kLwPlanFree = 32.0 * 1024 * 1024;

// Whether an analysis gets a plan, with which the level walk is the default shape
// of an ORDER or MULTIROW solve with one right-hand side.
bool level_walk_fits(const sp_mat_t* m, const dfr_analysis_info_t* info) {
    if (!info || !info->iorder || !info->inv_iorder || !info->bucket_off || !info->level || info->nlevs < 1) return false;
    if (!m->priv || info->n != m->nr || m->nr < 1 || m->nnz > kLwMaxEntries || !analysis_id(info)) return false;
    const int longest = static_cast<const MatPriv*>(m->priv)->max_row - 1;
    if (longest > kLongRow || chain_of(m, info)) return false;
    const bool lane_rows = longest <= kLwU;
    return (12.0 * m->nnz + 32.0 * m->nr) / info->nlevs <= (lane_rows ? kLwShortLevelBytes : kLwLevelBytes);
}

static void free_level_plan(LevelPlan& L) {
    if (L.block) (void)hipFree(L.block);
    L = LevelPlan{};
}

// A matrix's plans are looked up and released under this lock: a thread that
// frees an analysis releases its plans in every live matrix.
static std::mutex g_lw_mu;

void drop_level_plans(MatPriv* pv) {
    std::lock_guard<std::mutex> g(g_lw_mu);
    for (auto& p : pv->lw) free_level_plan(p.second);
    pv->lw.clear();
}

void drop_level_plan(MatPriv* pv, unsigned long long id) {
    std::lock_guard<std::mutex> g(g_lw_mu);
    const auto it = pv->lw.find(id);
    if (it == pv->lw.end()) return;
    free_level_plan(it->second);
    pv->lw.erase(it);
}

// The plan for analysis `id` (map entries stay where they are).
static LevelPlan* find_level_plan(MatPriv* pv, unsigned long long id, bool make) {
    std::lock_guard<std::mutex> g(g_lw_mu);
    const auto it = pv->lw.find(id);
    if (it != pv->lw.end()) return &it->second;
    return make ? &pv->lw[id] : nullptr;
}

bool level_plan_made(const sp_mat_t* m, const dfr_analysis_info_t* info) {
    const unsigned long long id = analysis_id(info);
    const LevelPlan* L = id ? find_level_plan(static_cast<MatPriv*>(m->priv), id, false) : nullptr;
    return L && !L->bad && info->n == m->nr && level_walk_fits(m, info);
}

static unsigned lw_grid(long long threads) {
    return (unsigned)std::max<long long>(1, std::min<long long>((threads + 255) / 256, 8192));
}

// Waves of the workgroup: enough for a typical level's slices in one step.
static LwShape lw_shape(const sp_mat_t* m, const dfr_analysis_info_t* info) {
    const MatPriv* pv = static_cast<const MatPriv*>(m->priv);
    const double off = (double)(m->nnz - m->nr) / m->nr, rows = (double)m->nr / info->nlevs;
    const double lanes = off <= 4 ? 1 : off <= 8 ? 2 : off <= 16 ? 4 : 8;
    const double slices = rows * lanes / kWave;
    LwShape sh{};
    sh.nw = slices <= 0.75 ? 1 : slices <= 3 ? 4 : 8;
    const int longest = pv->max_row - 1;
    sh.lg_big = 3;
    while (sh.lg_big < 6 && (kLwU << sh.lg_big) < longest) ++sh.lg_big;
    return sh;
}

// Words of working memory to make a plan.
size_t level_plan_work(int nlevs) { return 2 * ((size_t)nlevs + 1) + 3 + scan_scratch((long long)nlevs + 1); }

// The plan: steps, slices, slots and the entry of each slot, with room for one
// solve's records.  work: level_plan_work words, or null to allocate them.
static int lw_structure(const sp_mat_t* m, const dfr_analysis_info_t* info, LevelPlan& L, int* work) {
    const int nl = info->nlevs, n = m->nr;
    const LwShape sh = lw_shape(m, info);
    L.nw = sh.nw;
    L.permuted = n > kLwInPlace;
    hipStream_t s = nullptr;
    int* own = nullptr;
    int st = SPTRSV_OK;
    auto chk = [&](hipError_t e, const char* what) {
        if (e != hipSuccess && st == SPTRSV_OK) st = hip_fail(e, what, __FILE__, __LINE__);
        return st == SPTRSV_OK;
    };
    auto build = [&]() {
        if (!work && !chk(hipMalloc(&own, sizeof(int) * level_plan_work(nl)), "level walk count")) return;
        int *slices = work ? work : own, *steps = slices + nl + 1, *flags = steps + nl + 1, *sums = flags + 3;
        hipLaunchKernelGGL(k_lw_count, dim3(lw_grid(nl + 1)), dim3(256), 0, s, info->bucket_off, nl, sh, slices, steps, flags);
        if (!chk(hipGetLastError(), "level walk count")) return;
        if ((st = exclusive_scan(slices, slices, (long long)nl + 1, s, sums)) != SPTRSV_OK) return;
        if ((st = exclusive_scan(steps, steps, (long long)nl + 1, s, sums)) != SPTRSV_OK) return;
        std::vector<int> h((size_t)nl + 2);  // both totals in one copy
        if (!chk(hipMemcpy(h.data(), slices + nl, sizeof(int) * h.size(), hipMemcpyDeviceToHost), "level walk count")) return;
        L.n_slices = h.front();
        L.nsteps = h.back();
        if (L.n_slices > kLwMaxSlices || (double)L.n_slices * kLwSliceBytes > kLwPlanShare * m->nnz + kLwPlanFree) {
            L.bad = true;
            return;
        }
        // whole blocks of 64 steps, and one of empty ones for the loads ahead
        L.n_steps_all = (L.nsteps + 63) / 64 * 64 + 64;
        const size_t slots = (size_t)L.n_slices * kWave;
        const int over_cap = 64 + L.n_slices / 4;
        int2* slice = nullptr;
        unsigned* step = nullptr;
        Arena ar;
        ar.add(&slice, L.n_slices);
        ar.add(&step, L.n_steps_all);
        ar.add(&L.col, slots * kLwU);
        ar.add(&L.from, slots * kLwU);
        ar.add(&L.fcol, slots);
        ar.add(&L.ffrom, slots);
        ar.add(&L.over, L.n_slices);
        ar.add(&L.ocol, (size_t)over_cap * kWave);
        ar.add(&L.ofrom, (size_t)over_cap * kWave);
        ar.add(&L.diag_from, n);
        ar.add(&L.order, n);
        // the records: sized for the widest ones (mixed), so that solves of every
        // precision use the same memory and none allocates; with all that far
        // entries and overflow lists can take, which is known only later (one
        // allocation: each costs an analysis some 20 us, its release as much)
        constexpr size_t rec_words = 3, row_words = 4;
        const bool may_far = lw_near(n - 1) > 0;
        ar.add(&L.rec, slots * kLwU * rec_words);
        ar.add(&L.frec, may_far ? slots * rec_words : 0);
        ar.add(&L.orec, (size_t)over_cap * kWave * rec_words);
        ar.add(&L.rows, slots * row_words);
        ar.add(&L.piv32, slots);
        ar.add(&L.pub, may_far ? n : 0);
        ar.add(&L.b, L.permuted ? n : 0);
        ar.add(&L.x, L.permuted ? n : 0);
        if (!chk(ar.get(&L.block), "level walk plan")) return;
        L.slice = slice;
        L.step = step;
        hipLaunchKernelGGL(k_lw_slices, dim3(lw_grid(nl)), dim3(256), 0, s, info->bucket_off, nl, sh, slices, steps,
                           L.n_steps_all, slice, step);
        hipLaunchKernelGGL(k_lw_slots, dim3(lw_grid((long long)slots)), dim3(256), 0, s, m->ia, m->ja, info->iorder,
                           info->inv_iorder, info->level, L.permuted, slice, L.n_slices, L.col, L.from, L.fcol, L.ffrom,
                           L.over, L.ocol, L.ofrom, over_cap, L.diag_from, L.order, flags);
        int f[3];
        if (!chk(hipGetLastError(), "level walk slots") ||
            !chk(hipMemcpy(f, flags, sizeof(f), hipMemcpyDeviceToHost), "level walk flags"))
            return;
        L.bad = f[0] != 0 || f[2] > kLwFarShare * m->nnz;
        L.n_over = f[1];
        L.far = f[2] > 0;
    };
    build();
    if (own) (void)hipFree(own);
    if (L.bad) {
        free_level_plan(L);
        L.bad = true;
    }
    return st;
}

// The plan for `info`, made when there is none yet.  *plan stays null where the
// walk cannot be taken: the stream is being captured before the plan exists
// (a solve that names the walk for a matrix whose analysis made none), there is
// no memory for the plan, or the analysis does not fit.  A plan that a
// solve has used (and a captured solve holds) stays until its analysis or its
// matrix goes.
static int lw_prepare(sp_mat_t* m, const dfr_analysis_info_t* info, hipStream_t s, const LevelPlan** plan,
                      int* work = nullptr) {
    MatPriv* pv = priv_of(m);
    *plan = nullptr;
    const unsigned long long id = analysis_id(info);
    if (!id || !info->iorder || !info->inv_iorder || !info->bucket_off || !info->level || info->n != m->nr ||
        info->nlevs < 1 || m->nnz > kLwMaxEntries)
        return SPTRSV_OK;
    const LevelPlan* have = find_level_plan(pv, id, false);
    if (have) {
        *plan = have->bad ? nullptr : have;
        return SPTRSV_OK;
    }
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return SPTRSV_OK;
    }
    LevelPlan& L = *find_level_plan(pv, id, true);
    const int st = lw_structure(m, info, L, work);
    if (st == SPTRSV_E_ALLOC) {
        (void)hipGetLastError();
        free_level_plan(L);
        L.bad = true;  // not tried again for this analysis
        return SPTRSV_OK;
    }
    if (st != SPTRSV_OK) {
        drop_level_plan(pv, id);
        return st;
    }
    *plan = L.bad ? nullptr : &L;
    return SPTRSV_OK;
}

int make_level_plan(sp_mat_t* m, const dfr_analysis_info_t* info, int* work) {
    const LevelPlan* plan = nullptr;
    return level_walk_fits(m, info) ? lw_prepare(m, info, nullptr, &plan, work) : SPTRSV_OK;
}

template <class P, int WG, int D>
static hipError_t lw_launch(const LwArgs& A, bool far, hipStream_t s) {
    if (far)
        hipLaunchKernelGGL((k_level_walk<P, WG, D, true>), dim3(1), dim3(WG), 0, s, A);
    else
        hipLaunchKernelGGL((k_level_walk<P, WG, D, false>), dim3(1), dim3(WG), 0, s, A);
    return hipGetLastError();
}

template <class P>
static int lw_run(sp_mat_t* m, dfr_analysis_info_t* info, const void* b, void* x, hipStream_t s, bool timed, bool* done) {
    constexpr bool f32 = std::is_same<P, PolF32>::value;
    const LevelPlan* plan = nullptr;
    SPT_TRY(lw_prepare(m, info, s, &plan));
    *done = plan != nullptr;
    if (!plan) return SPTRSV_OK;
    const LevelPlan& L = *plan;
    LwArgs A{};
    A.nsteps = L.nsteps;
    A.step = static_cast<const unsigned*>(L.step);
    A.rec = L.rec;
    A.frec = L.frec;
    A.rows = L.rows;
    A.piv32 = L.piv32;
    A.over = L.over;
    A.orec = L.orec;
    A.ocol = L.ocol;
    A.b = L.permuted ? L.b : b;
    A.x = L.permuted ? L.x : x;
    A.pub = L.pub;
    A.n = (unsigned)m->nr;
    A.n_steps_all = (unsigned)L.n_steps_all;
    A.n_slices = (unsigned)L.n_slices;
    const KtPair ev = timed ? kernel_timer_pair(s) : KtPair{};
    if (ev) SPT_HIP(hipEventRecord(ev[0], s));
    using T = typename std::conditional<f32, float, double>::type;
    LwFill<T> F{};
    F.slice = static_cast<const int2*>(L.slice);
    F.n_slices = L.n_slices;
    F.col = L.col;
    F.fcol = L.fcol;
    F.ocol = L.ocol;
    F.from = L.from;
    F.ffrom = L.ffrom;
    F.ofrom = L.ofrom;
    F.n_over_slots = (long long)L.n_over * kWave;
    F.over = L.over;
    F.order = L.order;
    F.diag_from = L.diag_from;
    if constexpr (f32) F.a = m->a32;
    else F.a = m->a;
    F.rec = L.rec;
    F.frec = L.far ? L.frec : nullptr;
    F.orec = L.orec;
    F.rowrec = L.rows;
    F.piv32 = L.piv32;
    F.b = static_cast<const T*>(b);
    F.bp = L.permuted ? reinterpret_cast<T*>(L.b) : nullptr;
    F.n = m->nr;
    hipLaunchKernelGGL((k_lw_fill<T, std::is_same<P, PolMixed>::value>), dim3(lw_grid((long long)L.n_slices * kWave)),
                       dim3(256), 0, s, F);
    SPT_HIP(hipGetLastError());
    const hipError_t e = L.nw == 1   ? lw_launch<P, 64, 4>(A, L.far, s)
                         : L.nw == 4 ? lw_launch<P, 256, 4>(A, L.far, s)
                                     : lw_launch<P, 512, 4>(A, L.far, s);
    if (e != hipSuccess) return hip_fail(e, "level walk launch", __FILE__, __LINE__);
    if (L.permuted) {
        hipLaunchKernelGGL(k_lw_scatter<T>, dim3(lw_grid(m->nr)), dim3(256), 0, s, reinterpret_cast<const T*>(L.x), L.order, m->nr,
                           static_cast<T*>(x));
        SPT_HIP(hipGetLastError());
    }
    if (ev) SPT_HIP(hipEventRecord(ev[1], s));
    return SPTRSV_OK;
}

int level_walk_f64(sp_mat_t* m, dfr_analysis_info_t* info, const void* b, void* x, hipStream_t s, bool timed, bool* done) {
    return lw_run<PolF64>(m, info, b, x, s, timed, done);
}
int level_walk_f32(sp_mat_t* m, dfr_analysis_info_t* info, const void* b, void* x, hipStream_t s, bool timed, bool* done) {
    return lw_run<PolF32>(m, info, b, x, s, timed, done);
}
int level_walk_mixed(sp_mat_t* m, dfr_analysis_info_t* info, const void* b, void* x, hipStream_t s, bool timed,
                     bool* done) {
    return lw_run<PolMixed>(m, info, b, x, s, timed, done);
}

}  // namespace sptrsv
