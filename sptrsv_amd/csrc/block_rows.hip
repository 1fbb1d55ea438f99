// block_rows.hip -- the block walk (variant 5): 64 consecutive rows per wave,
// one row per lane, dependencies inside the block resolved in registers.
//
// In natural order the row before is what a row of a banded matrix or of a grid
// waits for first.  Through memory that costs 0.65 to 0.8 us a row, and a walk
// with one row per wave has 8192 rows in flight, less than one plane of a large
// grid.  Here a solved row reaches the rest of its block with v_readlane, so a
// row costs 32 ns (banded kernel) or 165 ns (short rows), and 64 times as many
// rows are in flight.  What bounds it then is the chain of blocks: for a band,
// 64 steps and one hand-off through memory per block; for a grid, a hand-off
// per line of the grid.
//
// Measured (natural-order solve, before -> now): bandwidth 17, n = 50000 39.3 ->
// 2.13 ms, bandwidth 60 41 -> 2.43 ms; 3D grid 101^3 FP32 8.7 -> 0.57 ms, 31^3
// 216 -> 107 us; 2D grid 707^2 19.5 -> 1.41 ms, 200^2 657 -> 358 us, 64^2 130 ->
// 111 us.
#include <type_traits>

#include "syncfree.hpp"

namespace sptrsv {

constexpr int kBlkU = 4;    // entries of a lane loaded together
constexpr int kBlkRun = 8;  // rows solved between two publications

// How a policy keeps the coefficients of dependencies inside the block.
template <class P>
struct BlkOps {
    using V = double;
    __device__ static V pack(const typename P::Val& v) {
        if constexpr (std::is_same<P, PolMixed>::value) return v.v64;
        else return v.v;
    }
    __device__ static typename P::Val unpack(V v) {
        if constexpr (std::is_same<P, PolMixed>::value) return {(float)v, v};
        else return {v};
    }
};
template <>
struct BlkOps<PolF32> {
    using V = float;
    __device__ static V pack(const PolF32::Val& v) { return v.v; }
    __device__ static PolF32::Val unpack(V v) { return {v}; }
};

template <>
struct BlkOps<PolLevel> {
    using V = int;
    __device__ static PolLevel::Val unpack(V) { return {}; }
};

// The word a row's dependents in the block fold.  Only a published word has to
// differ from the unsolved pattern.
template <class P>
__device__ __forceinline__ typename P::word blk_word(const SolveArgs& A, const typename P::Diag& dg,
                                                     const typename P::Acc& t) {
    if constexpr (std::is_same<P, PolF64>::value) {
        return (uint64_t)__double_as_longlong(t.s * dg.piv);
    } else if constexpr (std::is_same<P, PolF32>::value) {
        return __float_as_uint(t.s * dg.piv);
    } else {
        typename P::Out o{};
        return P::finish(A, dg, t, o);
    }
}

// OR of v over the wave, wave-uniform.
__device__ __forceinline__ uint64_t wave_or(uint64_t v) {
    for (int s = 0; s < 6; ++s) v = lane_combine(v, s, [](uint64_t x, uint64_t y) { return x | y; });
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
}

// First row of this wave's block: blocks are handed out in start order.
__device__ __forceinline__ int claim_rows(const SolveArgs& A) {
    int t = 0;
    if (threadIdx.x == 0) t = atomicAdd(A.ticket, 1);
    return __builtin_amdgcn_readfirstlane(t) * kWave;
}

// Rows of at most U off-diagonals: a lane holds all of its row's entries, so a
// row is folded in storage order once the last one is there, whatever order
// they came in, and the rows of a block are solved in the order they get ready
// (a block may hold the end of one grid line and the start of the next, which
// do not wait for each other).  The polls of a turn are in flight while ready
// rows are solved; a turn solves at most kBlkRun of them one after the other,
// so that what arrived meanwhile is seen (1 turn 12 % slower, 2 to 8 alike).
template <class P, int U>
__global__ __launch_bounds__(64) void k_block_short(SolveArgs A) {
    using word = typename P::word;
    using Acc = typename P::Acc;
    using Val = typename P::Val;
    const int lane = threadIdx.x;
    const int base = claim_rows(A);
    if (base >= A.n) return;
    const int row = base + lane;
    const bool live = row < A.n;
    word* gpub = static_cast<word*>(A.pub);
    int p = 0, dpos = 0;
    if (live) {
        p = A.ia[row];
        dpos = A.ia[row + 1] - 1;
    }
    int col[U], local[U];  // the column, and its lane if it is in the block
    Val val[U] = {};
    word got[U] = {};
    unsigned pend = 0;     // entries outside the block still waited for
    int need = live ? 0 : -1;  // entries still waited for; -1: row solved
    uint64_t bits = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        col[u] = 0;
        local[u] = -1;
        if (p + u < dpos) {
            col[u] = A.ja[p + u];
            val[u] = P::load(A, p + u);
        }
    }
    const Acc seed = live ? P::seed(A, (size_t)row) : P::zero();
    typename P::Diag dg{};
    if (live) dg = P::diag(A, dpos);
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (p + u < dpos) {
            ++need;
            if (col[u] >= base && col[u] < row) {
                local[u] = col[u] - base;
                bits |= 1ull << local[u];
            } else {
                pend |= 1u << u;
            }
        }
    const uint64_t used = wave_or(bits);  // rows of the block that others of it depend on
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): no step below waits for these loads
    const long long t0 = wall_clock64();
    bool expired = false;
    int spins = 0;
    while (true) {
        // polls go out first, and are looked at after the rows that are ready
        const bool polls = __ballot(pend != 0) != 0;
        word w[U];
        if (polls) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                w[u] = P::kUnsolved;
                if ((pend >> u) & 1) w[u] = poll_global(&gpub[col[u]]);
            }
        }
        uint64_t ready = __ballot(need == 0);
        for (int turn = polls ? kBlkRun : kWave; ready && turn; --turn) {
            // the entries after the first in a sum of their own: 0.82 of the
            // rounding error of a row per wave with 8 entries (1.27 in one sum)
            Acc t = seed, rest = P::zero();
            P::fold(t, val[0], got[0]);  // 0 * 0 where there is no entry
#pragma unroll
            for (int u = 1; u < U; ++u) P::fold(rest, val[u], got[u]);
            t = P::add(t, rest);
            const word mine = blk_word<P>(A, dg, t);
            if (need == 0) {
                typename P::Out o{};
                const word r = P::finish(A, dg, t, o);
                publish_global(&gpub[row], r);
                P::emit(A, (size_t)row, o, r);
                need = -1;
            }
            for (uint64_t m = ready & used; m; m &= m - 1) {
                const int j = __builtin_ctzll(m);
                const word wj = bcast(mine, j);
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (local[u] == j) {
                        got[u] = wj;
                        --need;
                    }
            }
            ready = __ballot(need == 0);
        }
        if (polls) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if ((pend >> u) & 1) {
                    if (w[u] == P::kUnsolved && expired) w[u] = P::kPoison;
                    if (w[u] != P::kUnsolved) {
                        got[u] = w[u];
                        pend &= ~(1u << u);
                        --need;
                    }
                }
        }
        if (!__ballot(need >= 0)) break;
        if (++spins == 512) {
            spins = 0;
            if (!expired && wall_clock64() - t0 > A.wd_ticks) {
                expired = true;
                if (lane == 0) atomicOr(A.err, 1);
            }
        }
    }
}

// Columns at most 63 rows back: only the block before is outside, the rows are
// taken in order, and both blocks' coefficients are dense in LDS (64 KB in FP64:
// two waves per CU, 512 blocks ahead of the chain).  A step is a multiply by the
// reciprocal diagonal, two readlanes, a multiply-add and an add; rows are
// published eight at a time.  A wave whose predecessor has published nothing yet sleeps
// between polls: 500 waves spinning made every hand-off slower (n = 50000 3.09
// -> 2.04 ms, with one sum a row).
// blocks (of several matrices in one): first row and the matrix's end row of
// each block, else the blocks of one matrix in order.
template <class P>
__global__ __launch_bounds__(64) void k_block_band(SolveArgs A, const int2* __restrict__ blocks) {
    using word = typename P::word;
    using Acc = typename P::Acc;
    using O = BlkOps<P>;
    constexpr bool LEVEL = std::is_same<P, PolLevel>::value;
    // [column][lane]: the block before, then this one
    __shared__ typename O::V coef[LEVEL ? 1 : 2 * kWave * kWave];
    const int lane = threadIdx.x;
    int base = claim_rows(A), end = A.n;
    if (blocks) {
        const int2 bk = blocks[base / kWave];
        base = bk.x;
        end = bk.y;
    }
    if (base >= end) return;
    const int row = base + lane, before = base - kWave;
    const bool live = row < end;
    word* gpub = static_cast<word*>(A.pub);
    int p = 0, dpos = 0;
    if (live) {
        p = A.ia[row];
        dpos = A.ia[row + 1] - 1;
    }
    const Acc seed = live ? P::seed(A, (size_t)row) : P::zero();
    typename P::Diag dg{};
    if (live) dg = P::diag(A, dpos);
    uint64_t bits[2] = {0, 0};  // columns of the two blocks this row depends on
    for (; __ballot(p < dpos); p += kBlkU) {
        int c[kBlkU];
        typename P::Val v[kBlkU];
#pragma unroll
        for (int u = 0; u < kBlkU; ++u) {
            c[u] = before;
            if (p + u < dpos) {
                c[u] = A.ja[p + u];
                v[u] = P::load(A, p + u);
            }
        }
#pragma unroll
        for (int u = 0; u < kBlkU; ++u) {
            const int j = c[u] - before;
            if (p + u < dpos && j >= 0 && c[u] < row) {
                uint64_t& b = j < kWave ? bits[0] : bits[1];
                const uint64_t bit = 1ull << (j & (kWave - 1));  // (no column comes twice in a row)
                if constexpr (!LEVEL) {
                    coef[j * kWave + lane] = O::pack(v[u]);
                }
                b |= bit;
            }
        }
    }
    const uint64_t used = wave_or(bits[0]), chain = wave_or(bits[1]);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): no step below waits for these loads
    const long long t0 = wall_clock64();
    bool expired = false;
    int spins = 0;
    word prev = P::kUnsolved;
    constexpr uint64_t run = (1ull << kBlkRun) - 1;
    // Four partial sums, by runs of kBlkRun columns, and the right-hand side added
    // to them: in one accumulator that starts from it, entry after entry, the
    // error grew with the bandwidth (1.5 times that of the lanes' tree of a row per
    // wave at bandwidth 17, 2.6 at 63; 0.77 and 0.75 so; a longer step: n = 50000,
    // bandwidth 17, 2.04 -> 2.14 ms).  Eight sums 2.27 ms and 0.69.  A row's only
    // entry is folded into the right-hand side, as in that tree.
    constexpr int kParts = LEVEL ? 1 : 4;
    const uint64_t deps = bits[0] | bits[1];
    const bool one = (deps & (deps - 1)) == 0;
    Acc part[kParts];
#pragma unroll
    for (int h = 0; h < kParts; ++h)
        part[h] = !LEVEL && one && ((deps >> (h * kBlkRun) | deps >> ((h + kParts) * kBlkRun)) & run) ? seed : P::zero();
    const Acc base_sum = one && deps ? P::zero() : seed;
    auto fold = [&](const Acc& x, typename O::V c, word w, bool mine) {
        Acc f = x;
        P::fold(f, O::unpack(c), w);
        return mine ? f : x;
    };
#pragma unroll
    for (int g = 0; g < kWave; g += kBlkRun) {
        const uint64_t want = used & (run << g);
        if (!want) continue;
        typename O::V c[kBlkRun] = {};
        if constexpr (!LEVEL) {
#pragma unroll
            for (int s = 0; s < kBlkRun; ++s) c[s] = coef[(g + s) * kWave + lane];
        }
        while (__ballot(prev == P::kUnsolved) & want) {
            if (prev == P::kUnsolved) prev = expired ? P::kPoison : poll_global(&gpub[before + lane]);
            if (!__ballot(prev != P::kUnsolved)) __builtin_amdgcn_s_sleep(16);
            if (++spins == 512) {
                spins = 0;
                if (!expired && wall_clock64() - t0 > A.wd_ticks) {
                    expired = true;
                    if (lane == 0) atomicOr(A.err, 1);
                }
            }
        }
        const unsigned b8 = (unsigned)(bits[0] >> g);
        Acc& own = part[g / kBlkRun % kParts];
#pragma unroll
        for (int s = 0; s < kBlkRun; ++s) own = fold(own, c[s], bcast(prev, g + s), (b8 >> s) & 1);
    }
#pragma unroll
    for (int g = 0; g < kWave; g += kBlkRun) {
        Acc& own = part[g / kBlkRun % kParts];
        // (the group before's last, as the chain has just come from it)
        Acc rest = base_sum;
        if constexpr (!LEVEL) {
            constexpr int k = kParts;
            const int h = g / kBlkRun;
            rest = P::add(P::add(rest, P::add(part[(h + 1) % k], part[(h + 2) % k])), part[(h + 3) % k]);
        }
        Acc t = LEVEL ? own : P::add(rest, own);
        if (chain & (run << g)) {
            typename O::V c[kBlkRun] = {};
            if constexpr (!LEVEL) {
#pragma unroll
                for (int s = 0; s < kBlkRun; ++s) c[s] = coef[(kWave + g + s) * kWave + lane];
            }
            const unsigned b8 = (unsigned)(bits[1] >> g);
#pragma unroll
            for (int s = 0; s < kBlkRun; ++s) {
                own = fold(own, c[s], bcast(blk_word<P>(A, dg, t), g + s), (b8 >> s) & 1);
                t = LEVEL ? own : P::add(rest, own);
            }
        }
        if (live && lane >= g && lane < g + kBlkRun) {
            typename P::Out x{};
            const word r = P::finish(A, dg, t, x);
            publish_global(&gpub[row], r);
            P::emit(A, (size_t)row, x, r);
        }
    }
}

template <class P>
hipError_t launch_block_rows(const SolveArgs& A, bool banded, int longest, hipStream_t s) {
    const dim3 grid(ceil_div(A.n, kWave)), wg(kWave);
    if (banded)
        hipLaunchKernelGGL((k_block_band<P>), grid, wg, 0, s, A, static_cast<const int2*>(nullptr));
    else if (longest <= kBlockRow / 2)
        hipLaunchKernelGGL((k_block_short<P, kBlockRow / 2>), grid, wg, A.dyn_lds, s, A);
    else if (longest <= kBlockRow)
        hipLaunchKernelGGL((k_block_short<P, kBlockRow>), grid, wg, A.dyn_lds, s, A);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
template <class P>
hipError_t launch_band_blocks(const SolveArgs& A, const int2* blocks, int count, hipStream_t s) {
    hipLaunchKernelGGL((k_block_band<P>), dim3((unsigned)count), dim3(kWave), 0, s, A, blocks);
    return hipGetLastError();
}
template hipError_t launch_band_blocks<PolF64>(const SolveArgs&, const int2*, int, hipStream_t);
template hipError_t launch_band_blocks<PolMixed>(const SolveArgs&, const int2*, int, hipStream_t);
template hipError_t launch_block_rows<PolF64>(const SolveArgs&, bool, int, hipStream_t);
template hipError_t launch_block_rows<PolF32>(const SolveArgs&, bool, int, hipStream_t);
template hipError_t launch_block_rows<PolMixed>(const SolveArgs&, bool, int, hipStream_t);
template hipError_t launch_block_rows<PolLevel>(const SolveArgs&, bool, int, hipStream_t);

}  // namespace sptrsv
