// Batched, persistent Newton-Raphson kernel on the block plan (see nr_block.hpp, blocks.hpp); compiled
// once per value type and block size (nr_block_*.hip).
//
// One workgroup runs whole NR loops for G interleaved instances taken from a work queue; lane t serves
// instance t % G as slot t / G. Per iteration, separated by workgroup barriers:
//   assembly   by Ybus rows: Ibus = Ybus V, F = V conj(Ibus) - Sbus (+ slack share), its inf-norm
//              (BaseAlgo.cpp:56-129), and J's 2 x 2 blocks (BaseNRAlgo.tpp:202-260) from the same products
//   factor     level by level: each block of the factor, and of the forward-solved right-hand side, is
//              a - sum L D U over its products (klu_refactor, KLUSolver.cpp:47-59); pivot blocks are
//              stored inverted
//   tail       dense LU of the trailing unknowns, and their solution
//   backward   level by level: x = D (y - sum U x') (klu_solve)
//   update     slack_absorbed, Va, Vm, V (BaseNRAlgo.tpp:138-158)
//
// What bounds it is latency: a chain of dependent levels per iteration, each a barrier apart, with one or two
// instances on a compute unit, and the instructions one wave issues between two barriers. Bus blocks instead
// of unknowns shorten the chain (2000 buses: 33 + 33 levels for 53 + 53) and cut the products 4.8 times. The
// units of a wave are a stream of its own with byte offsets and wave-uniform control, so a product takes no
// decoding, a team no selects and no level a table look-up. Against the scalar kernel (k_nr) it took the
// 2000-bus N-1 sweep (2128 outages) from 3.65 to 1.89 ms with FP32 and from 8.2 to 3.8 ms with FP64 factors,
// 1500 outages of 10 000 buses from 46.9 to 14.3 ms, 701 N-2 outages of 613 buses from 0.57 to 0.41 ms.
#pragma once

#include "nr_block.hpp"

#include "blocks.hpp"
#include "engine.hpp"
#include "nr_device.hpp"

#include <type_traits>

namespace {

using pfgpu::kBlkAddrMask;
using pfgpu::kBlkAhead;
using pfgpu::kBlkAssign;
using pfgpu::kBlkCols;
using pfgpu::kBlkEnd;
using pfgpu::kBlkIn2;
using pfgpu::kBlkInv;
using pfgpu::kBlkLead;
using pfgpu::kBlkLevel;
using pfgpu::kBlkTeamShift;
using pfgpu::kBlkTwo;
using pfgpu_block::BArgs;

static_assert(kMaxEdits == pfgpu_block::kEdits);

// v of the lane D lanes below (a sum towards the higher lanes: their last lane is the team's leader).
// Below 16: within rows of 16 lanes, by DPP; lanes whose source lies outside the row get 0. With LAST, in steps
// of 16 and 32 every lane gets the value of the last lane of the row (of the 32 lanes) below instead, which is
// the leader's own addend: row_bcast:15 and row_bcast:31.
template <int D, bool LAST>
constexpr int kDppBelow = D < 16 ? 0x110 + D : !LAST ? 0 : D == 16 ? 0x142 : 0x143;
template <int D, bool LAST>
__device__ __forceinline__ float from_below(float v) {
    const int x = __builtin_bit_cast(int, v);
    constexpr int dpp = kDppBelow<D, LAST>;
    if constexpr (dpp) return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, x, dpp, 0xf, 0xf, true));
    else return __shfl_up(v, D);
}
template <int D, bool LAST>
__device__ __forceinline__ double from_below(double v) {
    constexpr int dpp = kDppBelow<D, LAST>;
    if constexpr (dpp) {
        const long long b = __builtin_bit_cast(long long, v);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), dpp, 0xf, 0xf, true);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), dpp, 0xf, 0xf, true);
        return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
    } else {
        return __shfl_up(v, D);
    }
}
// Sums N values over teams of 2^lt lanes (stride G) into each team's last lane; lt is uniform.
template <int G, int N, typename FT>
__device__ __forceinline__ void team_last(FT (&v)[N], int lt) {
    auto add = [&](auto d) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] += from_below<decltype(d)::value, G == 1>(v[i]);
    };
    if (lt > 0) {
        add(std::integral_constant<int, G>{});
        if constexpr (2 * G <= 32) if (lt > 1) {
            add(std::integral_constant<int, 2 * G>{});
            if constexpr (4 * G <= 32) if (lt > 2) {
                add(std::integral_constant<int, 4 * G>{});
                if constexpr (8 * G <= 32) if (lt > 3) {
                    add(std::integral_constant<int, 8 * G>{});
                    if constexpr (16 * G <= 32) if (lt > 4) {
                        add(std::integral_constant<int, 16 * G>{});
                        if constexpr (32 * G <= 32) if (lt > 5) add(std::integral_constant<int, 32 * G>{});
                    }
                }
            }
        }
    }
}

// A copy of v in a register of its own from here on: the unit that v is a part of can then be loaded anew in
// place (left to itself the compiler copies parts of a unit where its load ends, and waits for it there).
__device__ __forceinline__ int copy_of(int v) {
    int w;
    asm volatile("v_mov_b32 %0, %1" : "=v"(w) : "v"(v));
    return w;
}

// Walks one wave through its units: `step(q)` works on the unit in q, loads the unit kBlkAhead further on
// into q and returns whether it was the wave's last one of the level. Four units are in flight in registers
// of their own (an unrolled ring: nothing is copied, so no load is waited for before its unit's turn).
// A wave without units at a level only keeps its barrier.
template <class Step>
__device__ __forceinline__ void walk_levels(const int4*& next, const unsigned long long* masks, int nl, Step step) {
    // through the scalar cache (uniform loads from the constant address space)
    typedef __attribute__((address_space(4))) const unsigned long long cst_u64;
    const cst_u64* const mask = (const cst_u64*)masks;
    static_assert(kBlkAhead == 4);
    int l = 0;
    unsigned long long m = nl > 0 ? mask[0] : 0ull;
    auto advance = [&]() {
        __syncthreads();
        ++l;
        m >>= 1;
        if ((l & 63) == 0 && l < nl) m = mask[l >> 6];
    };
    while (l < nl && !(m & 1)) advance();
    if (l >= nl) return;
    // in this order, so that waiting for one leaves the later ones in flight
    int4 q0 = next[0];
    __builtin_amdgcn_sched_barrier(0);
    int4 q1 = next[64];
    __builtin_amdgcn_sched_barrier(0);
    int4 q2 = next[128];
    __builtin_amdgcn_sched_barrier(0);
    int4 q3 = next[192];
    __builtin_amdgcn_sched_barrier(0);
    next += 256;
    auto turn = [&](int4& q) {
        if (step(q)) {
            do advance();
            while (l < nl && !(m & 1));
        }
    };
    // one exit, after a whole turn of the ring: units past the wave's last one are padding that ends no task
    do {
        turn(q0);
        turn(q1);
        turn(q2);
        turn(q3);
    } while (l < nl);
}

// Workgroup state in dynamic LDS (pfgpu_block::state_bytes).
template <int G>
struct WgState {
    lds_dbl *part, *slack, *flast, *dval;
    lds_int *done, *it, *status, *piv, *grow, *dent, *drow, *nd, *d0, *ndone, *grp;
    __device__ __forceinline__ WgState(lds_u8* at, int NT) {
        part = (lds_dbl*)at;
        slack = part + NT / 64 * G;
        flast = slack + G;
        dval = flast + G;
        done = (lds_int*)(dval + G * kMaxEdits * 2);
        it = done + G;
        status = it + G;
        piv = status + G;
        grow = piv + G;
        dent = grow + G;
        drow = dent + G * kMaxEdits;
        nd = drow + G * kMaxEdits;
        d0 = nd + G;
        ndone = d0 + G;
        grp = ndone + 1;
    }
};

// The kernel's arguments where the launch left them (the phases out of line read them there).
typedef __attribute__((address_space(4))) const BArgs cargs;

// One instance's value pairs: the first nlds in LDS, the rest in the workgroup's spill area.
template <typename FT, int G, bool LEAN>
struct Values {
    typedef FT ft2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) FT lds_ft;
    typedef __attribute__((address_space(3))) ft2 lds_ft2;  // every LDS access is a ds_read / ds_write
    lds_ft2* Pl;  // pair q of instance g at q * G + g
    ft2* Pg;
    int nlds, g;
    __device__ __forceinline__ ft2 ld1(int q) const {
        if (LEAN || q < nlds) return Pl[q * G + g];
        return Pg[(size_t)(q - nlds) * G + g];
    }
    __device__ __forceinline__ void st1(int q, ft2 p) const {
        if (LEAN || q < nlds) Pl[q * G + g] = p;
        else Pg[(size_t)(q - nlds) * G + g] = p;
    }
    // a block's pairs q, q + 1 (a block never straddles the end of the LDS part: the host cuts between blocks)
    __device__ __forceinline__ void st2(int q, ft2 p0, ft2 p1, bool two) const {
        if (LEAN || q < nlds) {
            Pl[q * G + g] = p0;
            if (two) Pl[(q + 1) * G + g] = p1;
        } else {
            ft2* const p = Pg + (size_t)(q - nlds) * G + g;
            if (G == 1 && two) {  // one store: scattered lanes take a cycle each
                typedef FT ft4 __attribute__((ext_vector_type(4), aligned(2 * sizeof(FT))));
                *(ft4*)p = ft4{p0.x, p0.y, p1.x, p1.y};
            } else {
                p[0] = p0;
                if (two) p[G] = p1;
            }
        }
    }
    // writes a block that is no pivot
    __device__ __forceinline__ void set(int e, FT v00, FT v01, FT v10, FT v11) const {
        const bool cols = e & kBlkCols, in2 = e & kBlkIn2;
        st2(e & kBlkAddrMask, ft2{v00, in2 ? (cols ? v10 : v01) : (FT)0}, ft2{cols ? v01 : v10, in2 ? v11 : (FT)0},
            e & kBlkTwo);
    }
    // Writes old - sum to the target of word e (p0, p1: its pairs; s00 .. s11 the sums by row and column).
    // fill: the J fill, with nothing to subtract. Pivot blocks are inverted: the LU of the 2 x 2 block on
    // its own diagonal, d0 = a00 and d1 = a11 - a10 a01 / d0.
    __device__ __forceinline__ void put(int e, ft2 p0, ft2 p1, FT s00, FT s01, FT s10, FT s11, bool fill, FT gtau,
                                        bool& bad, bool& grow) const {
        const bool cols = e & kBlkCols, in2 = e & kBlkIn2;
        ft2 v0, v1;
        v0.x = p0.x - s00;
        v0.y = in2 ? p0.y - (cols ? s10 : s01) : (FT)0;
        v1.x = p1.x - (cols ? s01 : s10);
        v1.y = in2 ? p1.y - s11 : (FT)0;
        if (e & kBlkInv) {
            bad |= bad_pivot(v0.x);
            if (!fill) grow |= fabs(v0.x) < gtau * fabs(p0.x);
            const FT r0 = pivot_recip(v0.x);
            const FT l = v1.x * r0, d1 = v1.y - l * v0.y;
            const FT r1 = pivot_recip(d1), t = v0.y * r1;
            if (in2) {
                bad |= bad_pivot(d1);
                grow |= fabs(d1) < gtau * fabs(p1.y);
            }
            v0.x = in2 ? r0 + r0 * t * l : r0;
            v0.y = in2 ? -r0 * t : (FT)0;
            v1.x = in2 ? -r1 * l : (FT)0;
            v1.y = in2 ? r1 : (FT)0;
        }
        st2(e & kBlkAddrMask, v0, v1, e & kBlkTwo);
    }
};

// One instance's Ybus edits (Y_inst = Y - dval at dpos): the first kMaxEdits in LDS (entries, rows,
// values), any further ones read from memory.
struct Edits {
    lds_int *ent, *row;
    lds_dbl* val;
    const int* dpos;    // all of them, CSC positions
    const double* dval;
    const int* y_ent;
    int nd, nnzY;
    int r[kMaxEdits];  // rows, in registers
    __device__ __forceinline__ void load() {
#pragma unroll
        for (int d = 0; d < kMaxEdits; ++d) r[d] = d < nd ? row[d] : INT_MIN;
    }
    // whether an edit lies in the row of bus b (with more than kMaxEdits: every row is taken as edited)
    __device__ __forceinline__ bool hit(int b) const {
        bool h = nd > kMaxEdits;
#pragma unroll
        for (int d = 0; d < kMaxEdits; ++d) h |= r[d] == b;
        return h;
    }
    // y of entry e with the edits applied
    __device__ __forceinline__ c64 apply(c64 y, int e) const {
        int id[kMaxEdits];
#pragma unroll
        for (int d = 0; d < kMaxEdits; ++d) id[d] = d < nd ? ent[d] : INT_MIN;
#pragma unroll
        for (int d = 0; d < kMaxEdits; ++d)
            if (id[d] == e) {
                y.re -= val[2 * d];
                y.im -= val[2 * d + 1];
            }
        for (int d = kMaxEdits; d < nd; ++d) {
            const int p = dpos[d];
            if ((unsigned)p >= (unsigned)nnzY || y_ent[p] != e) continue;
            y.re -= dval[2 * d];
            y.im -= dval[2 * d + 1];
        }
        return y;
    }
};

template <int G>
__device__ __forceinline__ Edits edits_of(cargs& a, const WgState<G>& st, int g, int nd, int d0) {
    Edits e;
    e.ent = st.dent + g * kMaxEdits;
    e.row = st.drow + g * kMaxEdits;
    e.val = st.dval + g * kMaxEdits * 2;
    e.dpos = a.dpos + d0;
    e.dval = a.dval + 2 * (size_t)d0;
    e.y_ent = a.y_ent;
    e.nd = nd;
    e.nnzY = a.nnzY;
    return e;
}

// ---- assembly: one lane per Ybus row. With t = y V_c and s = V_r conj(t), the row's current is the sum of
// its t, its power S_r = V_r conj(I_r) that of its s, and J's block of an entry is
//   dS/dVa = -j s (+ j S_r on the diagonal),  |V_c| dS/dVm = s (+ S_r on the diagonal):
// the columns of |V| are scaled by |V| (their unknown is dVm / Vm), which takes no square root or division.
// Rows come longest first as jagged diagonals, so a wave's rows are of nearly one length, kEll entries at a
// time with their loads issued before the first is used; every second batch of rows is dealt in reverse, so
// that the lanes' sums are even. Returns the lane's largest |F|; bad, grow: pivots with nothing to eliminate.
template <typename FT, int G, int NT, bool LEAN, typename VL>
__device__ __forceinline__ double assemble(cargs& a, const Values<FT, G, LEAN>& X, const double* Y, const double* S,
                                           const double* V, VL Vl, bool v_lds, Edits ed, double sa, int s, bool& bad,
                                           bool& grow) {
    typedef typename Values<FT, G, LEAN>::ft2 ft2;
    typedef __attribute__((address_space(4))) const int cst_int;
    constexpr int nslot = NT / G;
    const FT gtau = (FT)a.growth_tau;
    const cst_int* const jd_ptr = (const cst_int*)a.jd_ptr;
    auto Vat = [&](int b) -> c64 {
        if (v_lds) return {Vl[2 * b * G], Vl[2 * b * G + 1]};
        return ld_c(V, b);
    };
    ed.load();
    const bool newton = !a.fdpf;
    for (int i = s; i < a.njc; i += nslot) {  // constant blocks
        const double* v = a.jc_val + 4 * i;
        const int e = a.jc_dst[i];
        const bool cols = e & kBlkCols;
        const FT f00 = (FT)v[0], f01 = (FT)v[1], f10 = (FT)v[2], f11 = (FT)v[3];
        X.put(e, ft2{f00, cols ? f10 : f01}, ft2{cols ? f01 : f10, f11}, (FT)0, (FT)0, (FT)0, (FT)0, true, gtau, bad, grow);
    }
    double fm = 0.0;
    const int nrow = a.nrow, njd = a.njd;
    for (int b0 = 0, odd = 0; b0 < nrow; b0 += nslot, odd ^= 1) {
        const int i = b0 + (odd ? nslot - 1 - s : s);
        if (i >= nrow) continue;
        int2 jd[kEll];
        c64 y[kEll];
        int ent[kEll];
        bool in[kEll];
        auto load = [&](int k0) {
#pragma unroll
            for (int u = 0; u < kEll; ++u) {
                const int k = min(k0 + u, njd - 1), at = jd_ptr[max(k, 0)];
                in[u] = k0 + u < njd && i < jd_ptr[max(k, 0) + 1] - at;
                ent[u] = in[u] ? at + i : 0;
                jd[u] = a.jd[ent[u]];
                y[u] = a.Yjd ? ld_c(a.Yjd, ent[u]) : ld_c(Y, a.jd_pos[ent[u]]);
            }
        };
        const int4 rw = a.rows[i];
        const c64 yd0 = a.Yrow ? ld_c(a.Yrow, i) : ld_c(Y, rw.z);
        load(0);
        const c64 vr = Vat(rw.x), sr = ld_c(S, rw.x);
        const double wr = (a.single_slack && newton) ? 0.0 : a.w[rw.x];
        const bool hit = ed.hit(rw.x);
        const c64 yd = hit ? ed.apply(yd0, a.nent + i) : yd0;
        c64 cur = cmul(yd, vr);
        const c64 sd = cmul(vr, cconj(cur));
        for (int k0 = 0;;) {
            c64 vc[kEll];
#pragma unroll
            for (int u = 0; u < kEll; ++u) vc[u] = Vat(jd[u].x);
            if (hit) {
#pragma unroll
                for (int u = 0; u < kEll; ++u) y[u] = ed.apply(y[u], ent[u]);
            }
#pragma unroll
            for (int u = 0; u < kEll; ++u) {
                if (!in[u]) continue;
                const c64 t = cmul(y[u], vc[u]), sv = cmul(vr, cconj(t));
                cur = cadd(cur, t);
                if (newton && jd[u].y != -1) X.set(jd[u].y, (FT)sv.im, (FT)sv.re, (FT)-sv.re, (FT)sv.im);
            }
            k0 += kEll;
            if (k0 >= njd || i >= jd_ptr[k0 + 1] - jd_ptr[k0]) break;
            load(k0);
        }
        const c64 pw = cmul(vr, cconj(cur));
        if (newton && rw.w != -1) {
            const FT v00 = (FT)(sd.im - pw.im), v01 = (FT)(sd.re + pw.re), v10 = (FT)(pw.re - sd.re), v11 = (FT)(sd.im + pw.im);
            X.put(rw.w, ft2{v00, v01}, ft2{v10, v11}, (FT)0, (FT)0, (FT)0, (FT)0, true, gtau, bad, grow);
        }
        c64 mis = csub(pw, sr);
        if (!a.single_slack || a.fdpf) mis.re += sa * wr;
        if (a.fdpf) {  // P and Q of the fast-decoupled method: the mismatch divided by |V|
            const double ivm = 1.0 / sqrt(vr.re * vr.re + vr.im * vr.im);
            mis.re *= ivm;
            mis.im *= ivm;
        }
        const bool two = rw.y & kBlkIn2;
        fm = fmax(fm, inf_if_nonfinite(fabs(mis.re)));
        if (two) fm = fmax(fm, inf_if_nonfinite(fabs(mis.im)));
        X.st1(rw.y & kBlkAddrMask, ft2{(FT)mis.re, two ? (FT)mis.im : (FT)0});
    }
    return fm;
}

// J's values in the reference's order at the voltages V (the matrix of the last linear solve).
template <int G, int NT>
__device__ __noinline__ void capture_j(cargs* ap, const double* Y, const double* V, double* Jx, lds_u8* state, int nd, int d0) {
    constexpr int nslot = NT / G;
    cargs& a = *uniform(ap);
    const int g = threadIdx.x % G, s = threadIdx.x / G;
    Edits ed = edits_of<G>(a, WgState<G>(state, NT), g, nd, d0);
    ed.load();
    for (int i = s; i < a.njc; i += nslot) {
        const int4 j = a.jc_jidx[i];  // in the order 00, 01, 10, 11
        const double* v = a.jc_val + 4 * i;
        if (j.x >= 0) Jx[j.x] = v[0];
        if (j.y >= 0) Jx[j.y] = v[1];
        if (j.z >= 0) Jx[j.z] = v[2];
        if (j.w >= 0) Jx[j.w] = v[3];
    }
    if (a.fdpf) return;
    auto put = [&](int4 j, c64 dva, c64 dvm) {
        if (j.x >= 0) Jx[j.x] = dva.re;
        if (j.y >= 0) Jx[j.y] = dva.im;
        if (j.z >= 0) Jx[j.z] = dvm.re;
        if (j.w >= 0) Jx[j.w] = dvm.im;
    };
    auto scaled = [](c64 v, c64 vc) -> c64 {
        const double ic = 1.0 / sqrt(vc.re * vc.re + vc.im * vc.im);
        return {v.re * ic, v.im * ic};
    };
    for (int i = s; i < a.nrow; i += nslot) {
        const int4 rw = a.rows[i];
        const c64 vr = ld_c(V, rw.x);
        const bool hit = ed.hit(rw.x);
        c64 yd = ld_c(Y, rw.z);
        if (hit) yd = ed.apply(yd, a.nent + i);
        c64 cur = cmul(yd, vr);
        const c64 sd = cmul(vr, cconj(cur));
        for (int k = 0; k < a.njd && i < a.jd_ptr[k + 1] - a.jd_ptr[k]; ++k) {
            const int e = a.jd_ptr[k] + i;
            c64 y = ld_c(Y, a.jd_pos[e]);
            if (hit) y = ed.apply(y, e);
            const c64 vc = ld_c(V, a.jd[e].x), t = cmul(y, vc), sv = cmul(vr, cconj(t));
            cur = cadd(cur, t);
            put(a.jd_jidx[e], {sv.im, -sv.re}, scaled(sv, vc));
        }
        const c64 pw = cmul(vr, cconj(cur));
        put(a.row_jidx[i], {sd.im - pw.im, pw.re - sd.re}, scaled(cadd(sd, pw), vr));
    }
}

// One bus of the voltage update (BaseNRAlgo.tpp:138-151): Va and Vm (taken from V first in the single-slack
// form, BaseNRSingleSlackAlgo.tpp:131-132) minus the Newton step, dvm relative to Vm if `rel`, then V = Vm
// exp(j Va), which is written to memory and, if Vl is given, to LDS. Returns Vm. Out of line: inlined FP64
// atan2 / sincos raise the kernel's registers past 128.
template <typename VL>
__device__ __noinline__ double step_bus(double* V, VL Vl, bool v_lds, double* __restrict__ Va, double* __restrict__ Vm, int b,
                                        double dva, double dvm, bool rel, bool polar_first) {
    double va, vm;
    if (polar_first) {
        const double vr = V[2 * b], vi = V[2 * b + 1];
        va = atan2(vi, vr);
        vm = sqrt(vr * vr + vi * vi);
    } else {
        va = Va[b];
        vm = Vm[b];
    }
    va -= dva;
    vm -= rel ? dvm * vm : dvm;
    Va[b] = va;
    Vm[b] = vm;
    double sn, cs;
    sincos(va, &sn, &cs);
    const double re = vm * cs, im = vm * sn;
    V[2 * b] = re;
    V[2 * b + 1] = im;
    if (v_lds) {
        Vl[0] = re;
        Vl[1] = im;
    }
    return vm;
}

template <typename FT, int G, int NT, bool LEAN>
__global__ void __launch_bounds__(NT, 4) k_nr_block(const BArgs a) {
    constexpr int kWaves = NT / 64;
    constexpr int nslot = NT / G;
    typedef FT ft2 __attribute__((ext_vector_type(2)));
    extern __shared__ __align__(16) unsigned char lds_raw[];
    // explicit LDS address space: every access is a ds_read / ds_write
    typedef __attribute__((address_space(3))) FT lds_ft;
    typedef __attribute__((address_space(3))) ft2 lds_ft2;
    lds_ft2* const Pl = (lds_ft2*)(lds_raw);  // pair q of instance g at q * G + g
    const WgState<G> wst((lds_u8*)lds_raw + a.sh_off, NT);
    lds_dbl* const s_part = wst.part;
    lds_dbl* const s_slack = wst.slack;
    lds_dbl* const s_flast = wst.flast;  // mismatch of the current solve's last iteration
    lds_int* const s_done = wst.done;
    lds_int* const s_it = wst.it;
    lds_int* const s_status = wst.status;
    lds_int* const s_piv = wst.piv;
    lds_int* const s_grow = wst.grow;
    lds_int* const s_nd = wst.nd;
    lds_int* const s_d0 = wst.d0;
    lds_int* const s_ndone = wst.ndone;
    lds_int* const s_grp = wst.grp;
    cargs* const ap = (cargs*)__builtin_amdgcn_kernarg_segment_ptr();

    const int tid = threadIdx.x;
    const int g = tid % G, s = tid / G;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = a.n, nlds = a.nlds, m = a.m;
    const bool v_lds = a.v_off >= 0;
    const bool timing = a.phase_t != nullptr && blockIdx.x == 0 && tid == 0;
    unsigned long long t_ph = timing ? wall_clock64() : 0ull;
    auto tmark = [&](int ph) {
        if (timing) {
            const unsigned long long t = wall_clock64();
            a.phase_t[ph] += t - t_ph;
            t_ph = t;
        }
    };
    ft2* const Pg = reinterpret_cast<ft2*>(a.Xg) + (size_t)blockIdx.x * (size_t)a.nspill * G;
    const Values<FT, G, LEAN> X{Pl, Pg, nlds, g};
    // pairs by byte offset (of instance 0), as the units give it: below `lds_end` an LDS address (the
    // kernel has no static LDS: the host checks that the values start at address 0)
    constexpr int kPair = 2 * (int)sizeof(FT) * G;
    const int xg = g * 2 * (int)sizeof(FT), lds_end = nlds * kPair;
    auto lds2 = [&](int off, ft2& p0, ft2& p1) {
        const lds_ft2* const p = (lds_ft2*)(size_t)(unsigned)(off + xg);
        p0 = p[0];
        p1 = p[G];
    };
    auto lds1 = [&](int off) -> ft2 { return *(lds_ft2*)(size_t)(unsigned)(off + xg); };
    // N blocks by offset, from anywhere if `far`: then every lane reads both LDS and memory (its first pair,
    // where the other is wanted) and selects, all reads issued before the first is waited for. As branches,
    // the reads of both sides fill the same registers and the compiler waits for each before it issues the
    // next: three or four memory latencies in turn per unit instead of one (factor levels of the 10 000-bus
    // N-1 in FP32 9.1 -> 7.6 ms per workgroup, of the 2000-bus one in FP64 2.17 -> 1.9 ms).
    auto fetch = [&](bool far, const auto& off, auto& p) {
        constexpr int N = sizeof(p) / sizeof(p[0]);
        if (!far) {
#pragma unroll
            for (int i = 0; i < N; ++i) lds2(off[i], p[i][0], p[i][1]);
            return;
        }
        ft2 f[N][2];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const ft2* const q = (const ft2*)((const char*)Pg + (size_t)(unsigned)max(off[i] - lds_end, 0)) + g;
            f[i][0] = q[0];
            f[i][1] = q[G];
        }
#pragma unroll
        for (int i = 0; i < N; ++i) lds2(off[i] < lds_end ? off[i] : 0, p[i][0], p[i][1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                p[i][h].x = off[i] < lds_end ? p[i][h].x : f[i][h].x;
                p[i][h].y = off[i] < lds_end ? p[i][h].y : f[i][h].y;
            }
    };
    // the same of N single pairs
    auto fetch1 = [&](const auto& off, auto& p) {
        constexpr int N = sizeof(p) / sizeof(p[0]);
        ft2 f[N];
#pragma unroll
        for (int i = 0; i < N; ++i)
            f[i] = ((const ft2*)((const char*)Pg + (size_t)(unsigned)max(off[i] - lds_end, 0)))[g];
#pragma unroll
        for (int i = 0; i < N; ++i) p[i] = lds1(off[i] < lds_end ? off[i] : 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            p[i].x = off[i] < lds_end ? p[i].x : f[i].x;
            p[i].y = off[i] < lds_end ? p[i].y : f[i].y;
        }
    };
    bool bad = false;   // a zero or non-finite pivot met by this lane
    bool grow = false;  // a pivot that lost more than growth_tau of its value to cancellation
    const FT gtau = (FT)a.growth_tau;
    // the zero pairs are never written otherwise
    if (s == 0) {
        Pl[a.zpair * G + g] = ft2{(FT)0, (FT)0};
        Pl[(a.zpair + 1) * G + g] = ft2{(FT)0, (FT)0};
    }
    const int4* const f_units = a.fs + (size_t)a.f_at[wave] * 64 + (tid & 63);
    const int4* const b_units = a.bs + (size_t)a.b_at[wave] * 64 + (tid & 63);

    // Persistent workgroups: groups of G instances from a work queue (zeroed by the launch's first kernel).
    for (;;) {
    if (tid == 0) *s_grp = atomicAdd(a.queue, 1);
    __syncthreads();
    const long long grp = __builtin_amdgcn_readfirstlane(*s_grp);
    __syncthreads();
    if (grp >= a.ngroups) break;
    const long long inst = grp * G + g;
    const bool valid = inst < a.ninst;
    const long long ii = (long long)blockIdx.x * G + g;  // workspace row of this lane's instance
    const long long oi = valid ? (a.imap ? (long long)a.imap[inst] : inst) : 0;  // the caller's instance
    const double* Y = a.Yx + oi * a.y_stride;
    long long row = oi * a.chain;
    bool run = valid;  // this instance solves the current step (uniform over its lanes)
    const double* S = a.S + row * a.s_stride;
    double* V = a.V + row * 2 * (long long)n;
    double* Va = a.Va + ii * (long long)n;
    double* Vm = a.Vm + ii * (long long)n;
    lds_dbl* const Vl = (lds_dbl*)(lds_raw + (v_lds ? a.v_off : 0)) + 2 * g;
    // this instance's Ybus edits: the first kMaxEdits in LDS, any further ones read from memory
    if (s == 0) {
        s_nd[g] = 0;
        s_d0[g] = 0;
        if (a.dptr != nullptr && valid) {
            s_d0[g] = a.dptr[oi];
            s_nd[g] = a.dptr[oi + 1] - a.dptr[oi];
        }
    }
    __syncthreads();
    if (s < kMaxEdits && s < s_nd[g]) {
        const int k = s_d0[g] + s, p = a.dpos[k];
        const bool in = (unsigned)p < (unsigned)a.nnzY;
        wst.dent[g * kMaxEdits + s] = in ? a.y_ent[p] : INT_MIN;
        wst.drow[g * kMaxEdits + s] = in ? a.y_row[p] : INT_MIN;
        wst.dval[(g * kMaxEdits + s) * 2] = a.dval[2 * k];
        wst.dval[(g * kMaxEdits + s) * 2 + 1] = a.dval[2 * k + 1];
    }
    const int nd = s_nd[g], d0 = s_d0[g];
    bool alive = valid;  // chain mode: the chain has not failed yet
    for (int step = 0; step < a.chain; ++step) {
    row = oi * a.chain + step;
    run = alive && row < a.nrows;
    S = a.S + (run ? row : 0) * a.s_stride;
    V = a.V + (run ? row : 0) * 2 * (long long)n;
    if (run && step > 0)  // warm start from the previous step's V (own buses: no barrier)
        for (int b = s; b < n; b += nslot) {
            V[2 * b] = V[2 * b - 2 * (long long)n];
            V[2 * b + 1] = V[2 * b + 1 - 2 * (long long)n];
        }
    // ---- init: Va / Vm from V, slack_absorbed = Re(sum Sbus) (BaseNRAlgo.tpp:60,77-79)
    double ssum = 0.0;
    if (run) {
        polar_of(V, 1, Va, Vm, s, n, nslot);
        for (int b = s; b < n; b += nslot) {
            ssum += S[2 * b];
            if (v_lds) {
                Vl[2 * b * G] = V[2 * b];
                Vl[2 * b * G + 1] = V[2 * b + 1];
            }
        }
    }
#pragma unroll
    for (int o = G; o < 64; o <<= 1) ssum += __shfl_xor(ssum, o);
    {
        const int lane = tid & 63, wave = tid >> 6;
        if (lane < G) s_part[wave * G + lane] = ssum;
        __syncthreads();
        if (s == 0) {
            double t = 0;
            for (int k = 0; k < kWaves; ++k) t += s_part[k * G + g];
            s_slack[g] = t;
            s_it[g] = 0;
            s_status[g] = 0;
            s_piv[g] = 0;
            s_grow[g] = 0;
            s_flast[g] = INFINITY;
            s_done[g] = run ? 0 : 1;
        }
        __syncthreads();
    }

    tmark(5);
    bool act = false;
    for (;;) {
        // ---- assembly, convergence ------------------------------------------------------------------
        bad = grow = false;
        double fm = 0.0;
        act = run && !s_done[g];
        if (act)
            fm = assemble<FT, G, NT, LEAN>(*ap, X, Y, S, V, Vl, v_lds, edits_of<G>(*ap, wst, g, nd, d0), s_slack[g], s, bad,
                                           grow);
        tmark(0);
        fm = inst_reduce<G, NT, true>(fm, s_part);
        if (s == 0 && act) {
            s_flast[g] = fm;
            const int it = s_it[g];
            if (it > 0 && !(fm <= 1.7976931348623157e308)) { s_status[g] = 3; s_done[g] = 1; }
            else if (fm < a.tol) s_done[g] = 1;  // (at iteration 0 too)
            else if (it == 0 ? a.max_iter <= 0
                             : a.fdpf ? ((it & 1) == 0 && it / 2 >= a.max_iter) : it >= a.max_iter) {
                s_status[g] = 2;
                s_done[g] = 1;
            }
        }
        __syncthreads();
        tmark(5);
        if (tid == 0) {
            int k = 0;
            for (int i = 0; i < G; ++i) k += s_done[i];
            *s_ndone = k;
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(*s_ndone) == G) break;
        act = run && !s_done[g];
        if (s == 0 && act) s_it[g] += 1;

        // ---- factor + forward solve ----------------------------------------------------------------
        {
            FT c[4] = {(FT)0, (FT)0, (FT)0, (FT)0};  // sums 00, 01, 10, 11
            const int4* next = f_units;
            walk_levels(next, a.f_mask + (size_t)wave * a.f_words, a.nlev, [&](int4& q) -> bool {
                const int w = copy_of(q.w), wu = __builtin_amdgcn_readfirstlane(w);
                const bool far = !LEAN && wu < 0;  // an operand of the wave lies outside LDS
                auto product = [&](const auto& p) {
                    const ft2 l0 = p[0][0], l1 = p[0][1], u0 = p[1][0], u1 = p[1][1], d0 = p[2][0], d1 = p[2][1];
                    const FT t00 = l0.x * d0.x + l0.y * d1.x, t01 = l0.x * d0.y + l0.y * d1.y;
                    const FT t10 = l1.x * d0.x + l1.y * d1.x, t11 = l1.x * d0.y + l1.y * d1.y;
                    c[0] = fma(t01, u0.y, fma(t00, u0.x, c[0]));
                    c[1] = fma(t01, u1.y, fma(t00, u1.x, c[1]));
                    c[2] = fma(t11, u0.y, fma(t10, u0.x, c[2]));
                    c[3] = fma(t11, u1.y, fma(t10, u1.x, c[3]));
                };
                auto ahead = [&]() {
                    q = *next;
                    next += 64;
                };
                const bool end = wu & kBlkEnd;
                // the task's last unit: its target's old value is read along
                auto target = [&]() { return (w & kBlkAssign) ? a.zpair * kPair : (w & kBlkAddrMask) * kPair; };
                ft2 p[4][2];
                if constexpr (LEAN) {
                    lds2(q.x, p[0][0], p[0][1]);
                    lds2(q.y, p[1][0], p[1][1]);
                    lds2(q.z, p[2][0], p[2][1]);
                    ahead();
                    if (!end) {
                        product(p);
                        return false;
                    }
                    lds2(target(), p[3][0], p[3][1]);
                    product(p);
                } else if (!end) {
                    const int off[3] = {q.x, q.y, q.z};
                    ft2 o[3][2];
                    fetch(far, off, o);
                    ahead();
                    product(o);
                    return false;
                } else {
                    const int off[4] = {q.x, q.y, q.z, target()};
                    fetch(far, off, p);
                    ahead();
                    product(p);
                }
                const ft2 p0 = p[3][0], p1 = p[3][1];
                team_last<G>(c, (wu >> kBlkTeamShift) & 7);
                if (w & kBlkLead) X.put(w, p0, p1, c[0], c[1], c[2], c[3], false, gtau, bad, grow);
                c[0] = c[1] = c[2] = c[3] = (FT)0;
                return (wu & kBlkLevel) != 0;
            });
            // (lanes of an instance that is done walk along over what its last iteration left)
            if (act && bad) s_piv[g] = 1;
            if (act && grow) s_grow[g] = 1;
        }
        tmark(1);
        // ---- dense tail ---------------------------------------------------------------------------
        if (m > 0) tail_by_waves<TailPairs<G>, FT, G, NT>(m, a.tail_src, s_done, s_piv);
        __syncthreads();  // (without a tail too: s_piv of the walk, set after its last level's barrier)
        tmark(2);
        // zero / non-finite pivot: klu_factor failure on the first factorisation of a fresh solver
        // (KLUSolver.cpp:38-44), klu_refactor failure afterwards (:50-57)
        if (s == 0 && act && s_piv[g]) {
            s_status[g] = (a.fresh && s_it[g] == 1) ? 5 : 6;  // (FDPF: the first half-step)
            s_done[g] = 1;
        }
        __syncthreads();
        act = run && !s_done[g];

        // ---- backward solve: x = D (y - sum U x') ------------------------------------------------------
        {
            FT c[2] = {(FT)0, (FT)0};
            const int4* next = b_units;
            walk_levels(next, a.b_mask + (size_t)wave * a.b_words, a.nblev, [&](int4& q) -> bool {
                const int w = copy_of(q.w), wu = __builtin_amdgcn_readfirstlane(w), d = copy_of(q.z);
                auto product = [&](const ft2 u0, const ft2 u1, const ft2 x) {
                    const FT v0 = w < 0 ? u1.x : (FT)0, v1 = w < 0 ? u1.y : (FT)0;  // else not the block's
                    c[0] = fma(v0, x.y, fma(u0.x, x.x, c[0]));
                    c[1] = fma(v1, x.y, fma(u0.y, x.x, c[1]));
                };
                auto ahead = [&]() {
                    q = *next;
                    next += 64;
                };
                constexpr int kNext = kPair;  // a block's second pair
                const bool end = wu & kBlkEnd;
                const int to = (w & kBlkAddrMask) * kPair;
                ft2 p[6];
                if constexpr (LEAN) {
                    lds2(q.x, p[0], p[1]);
                    p[2] = lds1(q.y);
                    ahead();
                    if (!end) {
                        product(p[0], p[1], p[2]);
                        return false;
                    }
                    lds2(d, p[3], p[4]);
                    p[5] = lds1(to);
                    product(p[0], p[1], p[2]);
                } else if (!end) {
                    const int off[3] = {q.x, q.x + kNext, q.y};
                    ft2 o[3];
                    fetch1(off, o);
                    ahead();
                    product(o[0], o[1], o[2]);
                    return false;
                } else {
                    const int off[6] = {q.x, q.x + kNext, q.y, d, d + kNext, to};
                    fetch1(off, p);
                    ahead();
                    product(p[0], p[1], p[2]);
                }
                const ft2 d0 = p[3], d1 = p[4], y = p[5];
                team_last<G>(c, (wu >> kBlkTeamShift) & 7);
                if (w & kBlkLead) {
                    const FT v0 = y.x - c[0], v1 = y.y - c[1];
                    X.st1(w & kBlkAddrMask, ft2{d0.x * v0 + d0.y * v1, d1.x * v0 + d1.y * v1});
                }
                c[0] = c[1] = (FT)0;
                return (wu & kBlkLevel) != 0;
            });
        }

        tmark(3);
        // ---- voltage update ------------------------------------------------------------------------------
        double vmin = INFINITY;
        if (act) {
            if (s == 0 && a.slack_x >= 0) s_slack[g] -= (double)X.ld1(a.slack_x).x;
            const bool keep = a.Jx_last != nullptr && row == a.jx_row;
            // FDPF: the P half-step (odd s_it) moves the angles only, the Q half the magnitudes
            const bool pstep = !a.fdpf || (s_it[g] & 1) != 0, qstep = !a.fdpf || (s_it[g] & 1) == 0;
            for (int b = s; b < n; b += nslot) {
                const int x = a.bus_y[b];
                ft2 dx = {(FT)0, (FT)0};
                if (x >= 0 && b != a.slack_bus) dx = X.ld1(x & kBlkAddrMask);
                const double dva = pstep ? (double)dx.x : 0.0;
                const double dvm = (qstep && x >= 0 && (x & kBlkIn2)) ? (double)dx.y : 0.0;
                if (keep) {
                    a.Vprev[2 * b] = V[2 * b];
                    a.Vprev[2 * b + 1] = V[2 * b + 1];
                }
                vmin = fmin(vmin, step_bus(V, Vl + 2 * b * G, v_lds, Va, Vm, b, dva, dvm, !a.fdpf, a.single_slack != 0));
            }
        }
        vmin = inst_reduce<G, NT, false>(vmin, s_part);
        if (act && vmin < 0.0) polar_of(V, 1, Va, Vm, s, n, nslot);
        __syncthreads();
        tmark(4);
    }
    if (run && a.Jx_last != nullptr && row == a.jx_row && s_it[g] > 0)  // J of the last linear solve
        capture_j<G, NT>(ap, Y, s_status[g] == 5 || s_status[g] == 6 ? V : a.Vprev, a.Jx_last,
                         (lds_u8*)lds_raw + a.sh_off, nd, d0);
    // ---- end of the step: results of this row; a failed chain stops ----------------------------------------
    if (run) {
        if (s == 0) {
            const int stt = s_status[g];
            a.iters[row] = a.fdpf ? (s_it[g] + 1) / 2 : s_it[g];
            a.status[row] = stt;
            if (a.flags)
                a.flags[row] = (stt != 0 && s_flast[g] < a.stall_tol ? kFlagStall : 0) | (s_grow[g] ? kFlagGrowth : 0);
        }
        alive = s_status[g] == 0;
    } else if (valid && row < a.nrows) {  // a step after its chain's failure
        for (int b = s; b < n; b += nslot) {
            double* Vr = a.V + row * 2 * (long long)n;
            Vr[2 * b] = 0.0;
            Vr[2 * b + 1] = 0.0;
        }
        if (s == 0) {
            a.iters[row] = 0;
            a.status[row] = kStatusNotRun;
            if (a.flags) a.flags[row] = 0;
        }
    }
    __syncthreads();  // the next step rewrites the workgroup state
    }  // step
    }  // instance groups
}

template <typename FT, int NT, bool LEAN>
const void* variant(int G) {
    switch (G) {
        case 1: return (const void*)k_nr_block<FT, 1, NT, LEAN>;
        case 2: return (const void*)k_nr_block<FT, 2, NT, LEAN>;
        case 4: return (const void*)k_nr_block<FT, 4, NT, LEAN>;
        case 8: return (const void*)k_nr_block<FT, 8, NT, LEAN>;
        case 16: return (const void*)k_nr_block<FT, 16, NT, LEAN>;
        case 32: return (const void*)k_nr_block<FT, 32, NT, LEAN>;
        default: throw pfgpu_engine::ApiError(PFGPU_E_INVALID, "instances_per_wg must be 1, 2, 4, 8, 16 or 32");
    }
}

}  // namespace
