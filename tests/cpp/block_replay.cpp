// Test-only: serial CPU replay of the block plan (lightsim2grid_amd/csrc/blocks.cpp) and its lane
// streams, one instance, in the storage the HIP kernel uses: the phases of one Newton iteration with
// every unit, team and target word as the kernel reads them. Never part of the product library.
#include "../../lightsim2grid_amd/csrc/blocks.hpp"

#include <cmath>
#include <complex>
#include <cstring>
#include <limits>
#include <set>
#include <vector>

using namespace pfgpu;

namespace {
struct Blk { double v[2][2]; };
}  // namespace

extern "C" {

// Returns the iterations, or a negative value. info: {levels, backward levels, products, pairs, tail,
// conflicts}. Values start as NaN: a read of a place that nothing wrote shows.
int block_replay_solve(int n, const int* Yp, const int* Yi, const double* Yx, const double* Sbus, const int* slack_ids,
                       int nslack, const double* w, const int* pv, int npv, const int* pq, int npq, int single_slack,
                       double* V, int max_iter, double tol, int G, int waves, int by_life, int* status, int* info) {
    YbusPattern Y;
    Y.n = n;
    Y.p.assign(Yp, Yp + n + 1);
    Y.i.assign(Yi, Yi + Yp[n]);
    const JPattern J = build_jacobian_pattern(Y, slack_ids, nslack, w, pv, npv, pq, npq, single_slack != 0);
    if (!has_block_form(J)) return -1;
    const BlockPlan P = build_block_plan(Y, J, column_order(J), by_life ? kByLife : kByUse);
    const BlockStreams S = build_block_streams(P, G, waves, 8, P.npairs);
    const int m = P.m, ld = m + 1;
    int conflicts = 0;
    using C = std::complex<double>;
    auto y = [&](int q) { return C(Yx[2 * q], Yx[2 * q + 1]); };
    std::vector<C> U(n), I(n);
    std::vector<double> Va(n), Vm(n);
    double slack = 0;
    for (int b = 0; b < n; ++b) {
        U[b] = C(V[2 * b], V[2 * b + 1]);
        Va[b] = std::arg(U[b]);
        Vm[b] = std::abs(U[b]);
        slack += Sbus[2 * b];
    }
    std::vector<double> X(2 * (size_t)P.npairs, std::numeric_limits<double>::quiet_NaN());
    for (int k = 0; k < 4; ++k) X[2 * P.zpair + k] = 0.0;
    const double nan = std::numeric_limits<double>::quiet_NaN();
    auto store = [&](int word, const Blk& b) {
        const int a = word & kBlkAddrMask;
        const bool in = word & kBlkIn2, out = word & kBlkTwo, cols = word & kBlkCols;
        const bool r2 = cols || word & kBlkInv ? in : out, c2 = cols ? out : in;
        if (word & kBlkInv) {
            const double r0 = 1.0 / b.v[0][0];
            double d[4] = {r0, 0, 0, 0};
            if (r2) {
                const double l = b.v[1][0] * r0, r1 = 1.0 / (b.v[1][1] - l * b.v[0][1]), t = b.v[0][1] * r1;
                d[0] = r0 + r0 * t * l; d[1] = -r0 * t; d[2] = -r1 * l; d[3] = r1;
            }
            for (int k = 0; k < 4; ++k) X[2 * a + k] = d[k];
        } else if (word & kBlkCols) {
            for (int c = 0; c <= c2; ++c) { X[2 * (a + c)] = b.v[0][c]; X[2 * (a + c) + 1] = r2 ? b.v[1][c] : 0.0; }
        } else {
            for (int r = 0; r <= r2; ++r) { X[2 * (a + r)] = b.v[r][0]; X[2 * (a + r) + 1] = c2 ? b.v[r][1] : 0.0; }
        }
    };
    auto load = [&](int word) -> Blk {
        const int a = word & kBlkAddrMask;
        const bool in = word & kBlkIn2, out = word & kBlkTwo, cols = word & kBlkCols;
        const bool r2 = cols || word & kBlkInv ? in : out, c2 = cols ? out : in;
        Blk b{};
        for (int r = 0; r <= r2; ++r)
            for (int c = 0; c <= c2; ++c) b.v[r][c] = word & kBlkCols ? X[2 * (a + c) + r] : X[2 * (a + r) + c];
        return b;
    };
    auto mismatch = [&]() -> double {
        double f = 0;
        std::fill(I.begin(), I.end(), C(0, 0));
        for (int c = 0; c < n; ++c)
            for (int q = Yp[c]; q < Yp[c + 1]; ++q) I[Yi[q]] += y(q) * U[c];
        for (int b = 0; b < n; ++b) {
            const int fw = P.bus_y[b];
            if (fw == -1) continue;
            C mis = U[b] * std::conj(I[b]) - C(Sbus[2 * b], Sbus[2 * b + 1]);
            if (!single_slack) mis += slack * w[b];
            const bool two = fw & kBlkIn2;
            const int a = fw & kBlkAddrMask;
            f = std::max(f, std::fabs(mis.real()));
            if (two) f = std::max(f, std::fabs(mis.imag()));
            X[2 * a] = mis.real();
            X[2 * a + 1] = two ? mis.imag() : 0.0;
        }
        return f;
    };
    double f = mismatch();
    int it = 0;
    *status = f < tol ? 0 : 2;
    while (*status == 2 && it < max_iter) {
        ++it;
        std::fill(X.begin() + 2 * (size_t)P.fill_at, X.end(), nan);  // V lies there while J is assembled
        for (size_t k = 0; k < P.jc_dst.size(); ++k) {
            Blk b;
            std::memcpy(b.v, &P.jc_val[4 * k], sizeof(b.v));
            store(P.jc_dst[k], b);
        }
        // the assembly's blocks: off-diagonal s = V_r conj(y V_c); columns of |V| scaled by |V|
        for (size_t i = 0; i < P.row_len.size(); ++i) {
            const int r = P.rows[4 * i];
            if (P.rows[4 * i + 1] != P.bus_y[r]) ++conflicts;
            C Ir = y(P.rows[4 * i + 2]) * U[r];
            const C sd = U[r] * std::conj(Ir);
            for (int k = 0; k < P.row_len[i]; ++k) {
                const size_t e = (size_t)P.jd_ptr[k] + i;
                const C t = y(P.jd_pos[e]) * U[P.jd[2 * e]], s = U[r] * std::conj(t);
                Ir += t;
                if (P.jd[2 * e + 1] != -1) store(P.jd[2 * e + 1], Blk{{{s.imag(), s.real()}, {-s.real(), s.imag()}}});
            }
            const C Sr = U[r] * std::conj(Ir);
            if (P.rows[4 * i + 3] != -1)
                store(P.rows[4 * i + 3], Blk{{{sd.imag() - Sr.imag(), sd.real() + Sr.real()}, {Sr.real() - sd.real(), sd.imag() + Sr.imag()}}});
        }
        const int step = 2 * 8 * G;
        auto lanes_agree = [&](const int* u) {  // the lanes of all instances hold the same unit
            for (int k = 0; k < 64; ++k)
                for (int x = 0; x < 4; ++x) conflicts += u[4 * k + x] != u[4 * (k / G * G) + x];
        };
        std::vector<size_t> at(S.f_at.begin(), S.f_at.end());
        for (int l = 0; l < P.nlev; ++l) {
            std::set<int> written, read;
            std::vector<std::pair<int, Blk>> out;
            for (int wv = 0; wv < waves; ++wv) {
                if (!(S.f_mask[(size_t)wv * S.f_words + l / 64] >> (l % 64) & 1)) continue;
                std::vector<Blk> acc(64, Blk{});
                for (bool more = true; more;) {
                    const int* u = &S.fs[256 * at[wv]++];
                    lanes_agree(u);
                    const int ctl = u[3];
                    for (int k = 0; k < 64; k += G) {
                        const int* q = u + 4 * k;
                        if ((q[3] ^ ctl) & (kBlkEnd | kBlkLevel | 7 << kBlkTeamShift)) ++conflicts;
                        for (int x = 0; x < 3; ++x) read.insert(q[x] / step);
                        const double* L = &X[2 * (q[0] / step)];
                        const double* Uc = &X[2 * (q[1] / step)];
                        const double* D = &X[2 * (q[2] / step)];
                        for (int r = 0; r < 2; ++r) {
                            const double t0 = L[2 * r] * D[0] + L[2 * r + 1] * D[2], t1 = L[2 * r] * D[1] + L[2 * r + 1] * D[3];
                            for (int c = 0; c < 2; ++c) acc[k].v[r][c] += t0 * Uc[2 * c] + t1 * Uc[2 * c + 1];
                        }
                    }
                    if (ctl & kBlkEnd) {
                        const int T = 1 << (ctl >> kBlkTeamShift & 7);
                        if (T * G > 64) ++conflicts;
                        for (int k = 0; k < 64; k += G) {
                            const int e = u[4 * k + 3];
                            if (!(e & kBlkLead)) continue;
                            if ((k / G) % T != T - 1) ++conflicts;
                            Blk b = e & kBlkAssign ? Blk{} : load(e);
                            for (int i = 0; i < T; ++i)
                                for (int r = 0; r < 2; ++r)
                                    for (int c = 0; c < 2; ++c) b.v[r][c] -= acc[k - i * G].v[r][c];
                            if (!written.insert(e & kBlkAddrMask).second) ++conflicts;
                            out.push_back({e, b});
                        }
                        acc.assign(64, Blk{});
                    }
                    more = !(ctl & kBlkLevel);
                }
            }
            for (auto& o : out) {
                conflicts += read.count(o.first & kBlkAddrMask);  // written while read
                store(o.first, o.second);
            }
        }
        // dense tail
        std::vector<double> T((size_t)m * ld);
        for (int k = 0; k < m * ld; ++k) T[k] = X[P.tail_src[k]];
        for (int k = 0; k < m; ++k)
            for (int i = k + 1; i < m; ++i) {
                const double lik = T[i * ld + k] / T[k * ld + k];
                for (int j = k + 1; j <= m; ++j) T[i * ld + j] -= lik * T[k * ld + j];
            }
        for (int k = m - 1; k >= 0; --k) {
            double s = T[k * ld + m];
            for (int j = k + 1; j < m; ++j) s -= T[k * ld + j] * X[P.tail_src[j * ld + m]];
            X[P.tail_src[k * ld + m]] = s / T[k * ld + k];
        }
        at.assign(S.b_at.begin(), S.b_at.end());
        for (int l = 0; l < P.nblev; ++l)
            for (int wv = 0; wv < waves; ++wv) {
                if (!(S.b_mask[(size_t)wv * S.b_words + l / 64] >> (l % 64) & 1)) continue;
                std::vector<double> a0(64, 0), a1(64, 0);
                for (bool more = true; more;) {
                    const int* u = &S.bs[256 * at[wv]++];
                    lanes_agree(u);
                    const int ctl = u[3];
                    for (int k = 0; k < 64; k += G) {
                        const int* q = u + 4 * k;
                        const double* Uc = &X[2 * (q[0] / step)];
                        const double* x = &X[2 * (q[1] / step)];
                        const bool two = q[3] & kBlkWide;
                        a0[k] += Uc[0] * x[0] + (two ? Uc[2] * x[1] : 0.0);
                        a1[k] += Uc[1] * x[0] + (two ? Uc[3] * x[1] : 0.0);
                    }
                    if (ctl & kBlkEnd) {
                        const int T = 1 << (ctl >> kBlkTeamShift & 7);
                        for (int k = 0; k < 64; k += G) {
                            const int* q = u + 4 * k;
                            if (!(q[3] & kBlkLead)) continue;
                            double s0 = 0, s1 = 0;
                            for (int i = 0; i < T; ++i) { s0 += a0[k - i * G]; s1 += a1[k - i * G]; }
                            double* x = &X[2 * (q[3] & kBlkAddrMask)];
                            const double* D = &X[2 * (q[2] / step)];
                            const double v0 = x[0] - s0, v1 = x[1] - s1;
                            x[0] = D[0] * v0 + D[1] * v1;
                            x[1] = D[2] * v0 + D[3] * v1;
                        }
                        a0.assign(64, 0.0);
                        a1.assign(64, 0.0);
                    }
                    more = !(ctl & kBlkLevel);
                }
            }
        if (P.slack_x >= 0) slack -= X[2 * P.slack_x];
        for (int b = 0; b < n; ++b) {
            if (P.bus_y[b] < 0 || b == P.slack_bus) continue;
            const int a = P.bus_y[b] & kBlkAddrMask;
            if (single_slack) { Va[b] = std::arg(U[b]); Vm[b] = std::abs(U[b]); }
            Va[b] -= X[2 * a];
            if (P.bus_y[b] & kBlkIn2) Vm[b] -= X[2 * a + 1] * Vm[b];
            U[b] = std::polar(std::fabs(Vm[b]), Vm[b] < 0 ? Va[b] + M_PI : Va[b]);
            if (Vm[b] < 0) { Va[b] = std::arg(U[b]); Vm[b] = std::abs(U[b]); }
        }
        f = mismatch();
        if (!std::isfinite(f)) { *status = 3; break; }
        if (f < tol) *status = 0;
    }
    for (int b = 0; b < n; ++b) { V[2 * b] = U[b].real(); V[2 * b + 1] = U[b].imag(); }
    info[0] = P.nlev; info[1] = P.nblev; info[2] = (int)P.prods.size() / 3; info[3] = P.npairs; info[4] = m; info[5] = conflicts;
    return it;
}

}  // extern "C"
