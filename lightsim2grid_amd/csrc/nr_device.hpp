// Device code shared by the Newton-Raphson kernels: complex arithmetic, polar conversions, team
// sums, pivots and the dense tail.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

#include "blocks.hpp"

namespace {

constexpr int kMaxEdits = 8;  // Ybus edits per instance kept in LDS
constexpr int kEll = 4;  // Ybus row entries read at a time in the mismatch (column groups of its table)
typedef __attribute__((address_space(3))) double lds_dbl;
typedef __attribute__((address_space(3))) int lds_int;
typedef __attribute__((address_space(3))) unsigned char lds_u8;

// Per-row diagnostic flags written by the NR kernel (pfgpu_stats / the fallback passes):
constexpr int kFlagStall = 1;   // not converged, but the last mismatch is below the stall level
constexpr int kFlagGrowth = 2;  // a pivot lost more than the growth threshold to cancellation
constexpr int kStatusNotRun = 8;  // chain step after the chain's first failure (NotInitError)

struct c64 {
    double re, im;
};
__device__ __forceinline__ c64 cmul(c64 a, c64 b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ c64 cconj(c64 a) { return {a.re, -a.im}; }
__device__ __forceinline__ c64 csub(c64 a, c64 b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ c64 cadd(c64 a, c64 b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ c64 ld_c(const double* p, int i) { return {p[2 * i], p[2 * i + 1]}; }

// Reduce over the nslot lanes of one instance: shuffles inside the wave
// (lanes g, g+G, ... of a wave), then the kWaves partials through LDS.
template <int G, int NT, bool IS_MAX>
__device__ __forceinline__ double inst_reduce(double v, lds_dbl* part) {
    constexpr int kWaves = NT / 64;
#pragma unroll
    for (int o = G; o < 64; o <<= 1) {
        const double u = __shfl_xor(v, o);
        v = IS_MAX ? fmax(v, u) : fmin(v, u);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane < G) part[wave * G + lane] = v;
    __syncthreads();
    const int g = threadIdx.x % G;
    double r = part[g];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) r = IS_MAX ? fmax(r, part[k * G + g]) : fmin(r, part[k * G + g]);
    return r;
}

__device__ __forceinline__ double inf_if_nonfinite(double a) { return (a <= 1.7976931348623157e308) ? a : INFINITY; }

// Polar form of one lane's buses (b0, b0 + step, ...).
// Kept out of line: an inlined FP64 atan2 raises the NR kernel's register
// count past 128 VGPRs, which at 1024 lanes per workgroup means scratch spills
// in the factor loop.
// Va = arg(V), Vm = |V| (BaseNRAlgo.tpp:77-79, BaseNRSingleSlackAlgo.tpp:131-132)
// V holds bus b at V[2 b vs] (vs = 1 in global memory, G in LDS).
template <typename VP>
__device__ __noinline__ void polar_of(VP V, int vs, double* __restrict__ Va, double* __restrict__ Vm, int b0, int n,
                                      int step) {
    for (int b = b0; b < n; b += step) {
        const double vr = V[2 * b * vs], vi = V[2 * b * vs + 1];
        Va[b] = atan2(vi, vr);
        Vm[b] = sqrt(vr * vr + vi * vi);
    }
}
// One bus of the voltage update (BaseNRAlgo.tpp:138-151): Va and Vm (taken from V first in
// the single-slack form, BaseNRSingleSlackAlgo.tpp:131-132) minus the Newton step, then
// V = Vm exp(j Va); returns Vm.
template <typename VP>
__device__ __noinline__ double update_bus(VP V, int vs, double* __restrict__ Va, double* __restrict__ Vm, int b,
                                          double dva, double dvm, bool polar_first) {
    double va, vm;
    if (polar_first) {
        const double vr = V[2 * b * vs], vi = V[2 * b * vs + 1];
        va = atan2(vi, vr);
        vm = sqrt(vr * vr + vi * vi);
    } else {
        va = Va[b];
        vm = Vm[b];
    }
    va -= dva;
    vm -= dvm;
    Va[b] = va;
    Vm[b] = vm;
    double sn, cs;
    sincos(va, &sn, &cs);
    V[2 * b * vs] = vm * cs;
    V[2 * b * vs + 1] = vm * sn;
    return vm;
}

// Lane streams. Level l uses lanes [0, U) with K items per lane, item k of lane s
// at base + k * U + s. End word (forward: item.w, backward: item.z): bits 0-24
// slot, 25 assign (a fill-in entry: its slot held another value before), 26-28
// log2(team), 29 reciprocal, 30 end of task, 31 the lane's last item of the level
// (the lane loads nothing after it).
constexpr int kSC = 2;  // items per prefetch group of the general walk
constexpr int kHB = 4;  // items of a level loaded ahead, during the level before it (lean walk)
constexpr int kEnd = 1 << 30;
__device__ __forceinline__ int4 no_item() { return int4{-1, -1, 0, 0}; }

// Moves v from lane + D to each lane (D < 16: within a row of 16 lanes by DPP row_shl,
// no LDS traffic; lanes whose source is outside the row get 0).
template <int D>
__device__ __forceinline__ float lane_down(float v) {
    if constexpr (D < 16) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x100 + D, 0xF, 0xF, true));
    } else {
        return __shfl_down(v, D);
    }
}
template <int D>
__device__ __forceinline__ double lane_down(double v) {
    if constexpr (D < 16) {
        const long long b = __builtin_bit_cast(long long, v);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), 0x100 + D, 0xF, 0xF, true);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x100 + D, 0xF, 0xF, true);
        return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
    } else {
        return __shfl_down(v, D);
    }
}

// Sum over a team of 2^lt lanes (stride G, aligned to 2^lt * G) into its lowest lane.
// maxlt (uniform) bounds the steps; lanes of smaller teams drop the later steps by a
// select, not a branch. All lanes of a team share lt, so the lanes a leader reads are
// active and in its team.
template <int G, typename FT>
__device__ __forceinline__ FT team_sum(FT acc, int lt, int maxlt) {
    if (maxlt > 0) { const FT t = lane_down<1 * G>(acc); acc += lt > 0 ? t : (FT)0; }
    if constexpr (2 * G <= 32) if (maxlt > 1) { const FT t = lane_down<2 * G>(acc); acc += lt > 1 ? t : (FT)0; }
    if constexpr (4 * G <= 32) if (maxlt > 2) { const FT t = lane_down<4 * G>(acc); acc += lt > 2 ? t : (FT)0; }
    if constexpr (8 * G <= 32) if (maxlt > 3) { const FT t = lane_down<8 * G>(acc); acc += lt > 3 ? t : (FT)0; }
    if constexpr (16 * G <= 32) if (maxlt > 4) { const FT t = lane_down<16 * G>(acc); acc += lt > 4 ? t : (FT)0; }
    if constexpr (32 * G <= 32) if (maxlt > 5) { const FT t = lane_down<32 * G>(acc); acc += lt > 5 ? t : (FT)0; }
    return acc;
}

// Reciprocal of a pivot: the FP32 factor form uses the hardware reciprocal (1 ulp),
// the FP64 form an IEEE division.
__device__ __forceinline__ float pivot_recip(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ __forceinline__ double pivot_recip(double v) { return 1.0 / v; }
// v of lane `lane` (uniform over the wave) in every lane
__device__ __forceinline__ float lane_read(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ double lane_read(double v, int lane) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// zero or non-finite pivot (klu_refactor failure)
template <typename FT>
__device__ __forceinline__ bool bad_pivot(FT v) { return !(fabs(v) > (FT)0 && fabs(v) < (FT)INFINITY); }

// A pointer that is the same in every lane (one instance per workgroup), in scalar registers.
template <typename T>
__device__ __forceinline__ T* uniform(T* p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (T*)((unsigned long long)hi << 32 | lo);
}

// Where a tail's numbers lie: the FT at (row `lane`, column c) of instance g, in units of FT; column m is the
// right-hand side. On the block plan by a table, by columns of 64 lanes (2 pair + component); else as a tile,
// row-major, stride m + 1, from slot 0 on. Lanes past the rows name a number that is there.
template <int G>
struct TailPairs {
    typedef __attribute__((address_space(1))) const int* src_t;
    int m, g;
    src_t src;
    __device__ __forceinline__ int operator()(int, int c) const {
        const int x = src[c * 64];
        return (2 * G) * (x >> 1) + 2 * g + (x & 1);
    }
};
template <int G>
struct TailTile {
    typedef __attribute__((address_space(1))) const int* src_t;
    int m, g;
    src_t src;
    __device__ __forceinline__ int operator()(int lane, int c) const { return (min(lane, m - 1) * (m + 1) + c) * G + g; }
};

// ---------------------------------------------------------------------------
// Dense tail of one instance (m <= kMaxTail unknowns) on one wave, in registers: lane = row, R[j] = the j-th
// column that is left, Y = the right-hand side. A step eliminates the pivot's column from every other row,
// those above it too (Gauss-Jordan: their lanes are there anyway, and no backward sweep follows), and moves the
// columns one register down, so that it is a loop: unrolled over the pivots its FP64 form is 50 KB of code,
// which with the walks does not stay in the instruction cache. The pivot row reaches the other lanes by lane
// reads of each column, the next pivot's first, whose reciprocal is then formed beside the other columns'
// updates; no LDS access and no barrier lies between the pivots. A loop each for the last 8, 16, .. 48 columns.
// Where: where the numbers lie in LDS, from address 0 on; the right-hand side's places receive the solution.
// Returns whether a pivot was zero or non-finite.
// Bound by the instruction issue of one wave: about m^2 / 2 lane reads and as many updates. 43 unknowns of the
// 2000-bus grid, per iteration: 9.8 us in FP32, 15.6 in FP64 (two lane reads per value); two rows at a time to
// one of 16 waves in turn, a barrier and an LDS round trip per pair of pivots, it took 14 and 19 us. Unrolled it
// takes 1 us less, but the kernel is slower where factor levels are short (613-bus N-2: 437 against 410 us).
// With four instances per workgroup (118 buses, 4 waves) each wave takes one: 8 us instead of 15 for all four.
// Out of line: inlined, its registers and the walks' add up to spills in both.
// ---------------------------------------------------------------------------
template <int W, typename FT>
__device__ __forceinline__ void tail_steps(FT (&R)[pfgpu::kMaxTail], FT& Y, FT& D, FT& r, int& k, int m, int lane, bool& bad) {
    if constexpr (W > 0) {
        while (k < m && m - k > W - 8) {  // R[0 .. W - 1] hold what is left
            bad |= bad_pivot(lane_read(R[0], k));
            D = lane == k ? r : D;
            const FT l = lane == k ? (FT)0 : R[0] * r;
            const FT u0 = lane_read(R[1], k), uy = lane_read(Y, k);
            R[0] = R[1] - l * u0;
            r = pivot_recip(lane_read(R[0], k + 1));
            Y -= l * uy;
            // four lane reads, then four updates: a value just read by lane may not be used at once
#pragma unroll
            for (int j = 1; j + 1 < W; j += 4) {
                FT u[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (j + i + 1 < W) u[i] = lane_read(R[j + i + 1], k);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (j + i + 1 < W) R[j + i] = R[j + i + 1] - l * u[i];
                __builtin_amdgcn_sched_barrier(0);
            }
            ++k;
        }
        tail_steps<W - 8>(R, Y, D, r, k, m, lane, bad);
    }
}

template <class Where, typename FT>
__device__ __noinline__ bool tail_wave(int m_, int g_, const int* src_) {
    typedef __attribute__((address_space(3))) FT lds_ft;
    constexpr int M = pfgpu::kMaxTail;
    const int m = __builtin_amdgcn_readfirstlane(m_), g = __builtin_amdgcn_readfirstlane(g_);
    const int lane = threadIdx.x & 63;
    const Where where{m, g, (typename Where::src_t)(uniform((int*)src_) + lane)};
    auto at = [&](int i) -> lds_ft* { return (lds_ft*)(size_t)(unsigned)(i * (int)sizeof(FT)); };
    FT R[M], Y;
    int from[M];
    const int ys = where(lane, m);
#pragma unroll
    for (int c = 0; c < M; c += 8)
        if (c < m)
#pragma unroll
            for (int j = c; j < c + 8; ++j) from[j] = where(lane, min(j, m));
    Y = *at(ys);
#pragma unroll
    for (int c = 0; c < M; c += 8)
        if (c < m) {
#pragma unroll
            for (int j = c; j < c + 8; ++j) R[j] = *at(from[j]);
#pragma unroll
            for (int j = c; j < c + 8; ++j) R[j] = lane < m ? R[j] : (FT)0;
        }
    bool bad = false;
    FT D = (FT)0, r = pivot_recip(lane_read(R[0], 0));  // lane k: the reciprocal of pivot k; this pivot's
    int k = 0;
    tail_steps<M>(R, Y, D, r, k, m, lane, bad);
    if (lane < m) *at(ys) = Y * D;
    return bad;
}

// The tails of a workgroup's G instances (m <= kMaxTail), an instance to a wave.
template <class Where, typename FT, int G, int NT, typename LI>
__device__ __forceinline__ void tail_by_waves(int m, const int* src, LI done, LI piv) {
    for (int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); g < G; g += NT / 64) {
        if (done[g]) continue;
        if (tail_wave<Where, FT>(m, g, src)) piv[g] = 1;
    }
}

// ---- dense tail: the m x m tile of every instance ---------------------------------
// Tile at slots [0, m*(m+1)): row-major with row stride m + 1, the right-hand side
// held as column m. Right-looking LU with diagonal pivots, four columns per pass (one
// barrier per pass): pass k eliminates columns k .. k+c-1 (c = min(4, m - k)) from the
// trailing block (rows >= k+c, columns >= k+c, the vector included) with the rank-c update
//   T(i,j) -= sum_q L(i,k+q) U(k+q,j),
//   U(k+q,j) = T(k+q,j) - sum_{r<q} L(k+q,k+r) U(k+r,j),
//   L(i,k+q) = (T(i,k+q) - sum_{r<q} L(i,k+r) U(k+r,k+q)) / d_k+q,
// every lane computing the c x c diagonal block's factors and the L and U factors of its
// entry from the tile. Rows k+1 .. k+c-1 of U and the c reciprocal pivots are stored one
// pass later (so that no pass writes what it reads); L itself is not stored, nothing
// after the forward sweep reads it.
// Then the backward sweep on the first wave alone (its lanes hold s < 64 / G of
// every instance; LDS accesses of one wave complete in issue order, so its passes
// need no barrier): x_k = y_k / d_k, y_i -= U(i,k) x_k for i < k; with one instance per
// workgroup, in registers.
template <typename FT, int G, int NT, typename LP>
__device__ __forceinline__ void dense_tail_lds(LP Xl, int m, int g, int s, bool act, bool& bad) {
    constexpr int nslot = NT / G;
    const int ld = m + 1;
    auto T = [&](int i, int j) -> int { return (i * ld + j) * G + g; };  // LDS index
    // the previous pass's block: its columns, reciprocal pivots and L factors
    int pc = 0;
    FT pr0 = (FT)0, pr1 = (FT)0, pr2 = (FT)0, pr3 = (FT)0;
    FT pl10 = (FT)0, pl20 = (FT)0, pl21 = (FT)0, pl30 = (FT)0, pl31 = (FT)0, pl32 = (FT)0;
    for (int k = 0;; k += 4) {
        if (act) {
            const int c = min(4, m - k);  // columns of this pass's block (<= 0: none)
            FT r0 = (FT)0, r1 = (FT)0, r2 = (FT)0, r3 = (FT)0;
            FT l10 = (FT)0, l20 = (FT)0, l21 = (FT)0, l30 = (FT)0, l31 = (FT)0, l32 = (FT)0;
            if (c > 0) {
                // the block's LU, in the same order in every lane
                FT u01 = (FT)0, u02 = (FT)0, u03 = (FT)0, u12 = (FT)0, u13 = (FT)0, u23 = (FT)0;
                const FT d0 = Xl[T(k, k)];
                bad |= bad_pivot(d0);
                r0 = pivot_recip(d0);
                if (c > 1) {
                    u01 = Xl[T(k, k + 1)];
                    l10 = Xl[T(k + 1, k)] * r0;
                    const FT d1 = Xl[T(k + 1, k + 1)] - l10 * u01;
                    bad |= bad_pivot(d1);
                    r1 = pivot_recip(d1);
                }
                if (c > 2) {
                    u02 = Xl[T(k, k + 2)];
                    u12 = Xl[T(k + 1, k + 2)] - l10 * u02;
                    l20 = Xl[T(k + 2, k)] * r0;
                    l21 = (Xl[T(k + 2, k + 1)] - l20 * u01) * r1;
                    const FT d2 = Xl[T(k + 2, k + 2)] - l20 * u02 - l21 * u12;
                    bad |= bad_pivot(d2);
                    r2 = pivot_recip(d2);
                }
                if (c > 3) {
                    u03 = Xl[T(k, k + 3)];
                    u13 = Xl[T(k + 1, k + 3)] - l10 * u03;
                    u23 = Xl[T(k + 2, k + 3)] - l20 * u03 - l21 * u13;
                    l30 = Xl[T(k + 3, k)] * r0;
                    l31 = (Xl[T(k + 3, k + 1)] - l30 * u01) * r1;
                    l32 = (Xl[T(k + 3, k + 2)] - l30 * u02 - l31 * u12) * r2;
                    const FT d3 = Xl[T(k + 3, k + 3)] - l30 * u03 - l31 * u13 - l32 * u23;
                    bad |= bad_pivot(d3);
                    r3 = pivot_recip(d3);
                }
                // entries (i, j), i in [k+c, m), j in [k+c, m]: w rows of w + 1
                const int w = m - k - c, wc = w + 1;
                // row = floor((idx + 1/2) / wc): the fractional part of the exact
                // quotient stays >= 1/(2 wc) from an integer, far above the float error
                const float inv = __builtin_amdgcn_rcpf((float)wc);
                for (int idx = s; idx < w * wc; idx += nslot) {
                    const int rr = (int)(((float)idx + 0.5f) * inv);
                    const int i = k + c + rr, j = k + c + (idx - rr * wc);
                    const FT li0 = Xl[T(i, k)] * r0;
                    const FT u0j = Xl[T(k, j)];
                    FT upd = li0 * u0j;
                    if (c > 1) {
                        const FT li1 = (Xl[T(i, k + 1)] - li0 * u01) * r1;
                        const FT u1j = Xl[T(k + 1, j)] - l10 * u0j;
                        upd += li1 * u1j;
                        if (c > 2) {
                            const FT li2 = (Xl[T(i, k + 2)] - li0 * u02 - li1 * u12) * r2;
                            const FT u2j = Xl[T(k + 2, j)] - l20 * u0j - l21 * u1j;
                            upd += li2 * u2j;
                            if (c > 3) {
                                const FT li3 = (Xl[T(i, k + 3)] - li0 * u03 - li1 * u13 - li2 * u23) * r3;
                                const FT u3j = Xl[T(k + 3, j)] - l30 * u0j - l31 * u1j - l32 * u2j;
                                upd += li3 * u3j;
                            }
                        }
                    }
                    Xl[T(i, j)] -= upd;
                }
            }
            if (k >= 4 && pc > 1) {  // rows p+1 .. p+pc-1 of U of the previous pass's block
                const int p = k - 4;
                for (int j = p + 2 + s; j <= m; j += nslot) {
                    const FT u0j = Xl[T(p, j)];
                    const FT u1j = Xl[T(p + 1, j)] - pl10 * u0j;
                    Xl[T(p + 1, j)] = u1j;
                    if (pc > 2 && j > p + 2) {
                        const FT u2j = Xl[T(p + 2, j)] - pl20 * u0j - pl21 * u1j;
                        Xl[T(p + 2, j)] = u2j;
                        if (pc > 3 && j > p + 3)
                            Xl[T(p + 3, j)] = Xl[T(p + 3, j)] - pl30 * u0j - pl31 * u1j - pl32 * u2j;
                    }
                }
            }
            if (k >= 4 && pc > 0 && s == 0) {  // and its reciprocal pivots
                const int p = k - 4;
                Xl[T(p, p)] = pr0;
                if (pc > 1) Xl[T(p + 1, p + 1)] = pr1;
                if (pc > 2) Xl[T(p + 2, p + 2)] = pr2;
                if (pc > 3) Xl[T(p + 3, p + 3)] = pr3;
            }
            pc = max(c, 0);
            pr0 = r0; pr1 = r1; pr2 = r2; pr3 = r3;
            pl10 = l10; pl20 = l20; pl21 = l21; pl30 = l30; pl31 = l31; pl32 = l32;
        }
        __syncthreads();
        if (k >= m) break;
    }
    if (G == 1 && m <= 128) {
        // One instance per workgroup: lane s of the first wave holds y_s and y_s+64 in
        // registers, and x_k = y_k / d_k reaches every lane by a lane read of its owner,
        // so a step is a few dependent register operations. U(i, k) and 1/d_k are not
        // written by the sweep: each step's reads are issued one step ahead.
        if (threadIdx.x < 64 && act) {
            FT y0 = s < m ? Xl[T(s, m)] : (FT)0, y1 = s + 64 < m ? Xl[T(s + 64, m)] : (FT)0;
            // column k's reads, clamped into the tile (a lane's U entries of rows i >= k
            // are read but not used)
            auto col = [&](int k, FT& u0, FT& u1, FT& dk) {
                const int c = max(k, 0);
                dk = Xl[T(c, c)];
                u0 = Xl[T(min(s, m - 1), c)];
                u1 = Xl[T(min(s + 64, m - 1), c)];
            };
            FT u0, u1, dk;
            col(m - 1, u0, u1, dk);
            for (int k = m - 1; k >= 0; --k) {
                FT nu0, nu1, ndk;
                col(k - 1, nu0, nu1, ndk);
                const FT xk = lane_read(k < 64 ? y0 : y1, k & 63) * dk;
                if (s == (k & 63)) {
                    if (k < 64) y0 = xk;
                    else y1 = xk;
                }
                if (s < k) y0 -= u0 * xk;  // rows i < k only: a non-finite x_k leaves the others
                if (s + 64 < k) y1 -= u1 * xk;
                u0 = nu0; u1 = nu1; dk = ndk;
            }
            if (s < m) Xl[T(s, m)] = y0;
            if (s + 64 < m) Xl[T(s + 64, m)] = y1;
        }
    } else if (threadIdx.x < 64 && act) {
        constexpr int ws = 64 / G;  // lanes of one instance in the first wave
        for (int k = m - 1; k >= 0; --k) {
            const FT xk = Xl[T(k, m)] * Xl[T(k, k)];
            for (int i = s; i < k; i += ws) Xl[T(i, m)] -= Xl[T(i, k)] * xk;
            if (s == 0) Xl[T(k, m)] = xk;
            // keep this pass's LDS writes ahead of the next pass's reads in the code
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
}

}  // namespace
