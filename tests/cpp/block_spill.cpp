// Test-only: the addresses that the kernel forms on the units of a launch which spills (lightsim2grid_amd/csrc/
// blocks.cpp), checked one by one on the CPU for every cut between LDS and the spill area that is asked for. Never
// part of the product library.
#include "../../lightsim2grid_amd/csrc/blocks.hpp"

#include <algorithm>
#include <set>

using namespace pfgpu;

extern "C" {

// Cuts the values of a plan where `rooms` pairs of room put it and checks every unit of both walks; all_const: with
// a constant J (fast-decoupled grids). Returns the number of faults; info: {pairs, pairs fixed in LDS, cuts that
// spill, units marked as reaching outside LDS, unmarked units, J entries without a place or with two}.
int block_spill_check(int n, const int* Yp, const int* Yi, const int* slack_ids, int nslack, const double* w,
                      const int* pv, int npv, const int* pq, int npq, int single_slack, int all_const, int G, int waves,
                      int fsize, int nrooms, const int* rooms, int* info) {
    YbusPattern Y;
    Y.n = n;
    Y.p.assign(Yp, Yp + n + 1);
    Y.i.assign(Yi, Yi + Yp[n]);
    JPattern J = build_jacobian_pattern(Y, slack_ids, nslack, w, pv, npv, pq, npq, single_slack != 0);
    if (all_const) {
        std::fill(J.sel.begin(), J.sel.end(), (uint8_t)SEL_CONST);
        for (size_t q = 0; q < J.cval.size(); ++q) J.cval[q] = 1.0 + (double)q;
    }
    const BlockPlan P = build_block_plan(Y, J, column_order(J));
    int faults = 0;
    std::fill(info, info + 6, 0);
    info[0] = P.npairs;
    info[1] = P.fixed_pairs;
    // every J entry has one place: a constant block's or a row's
    std::vector<int> placed(J.Ji.size(), 0);
    for (const auto* v : {&P.jc_jidx, &P.jd_jidx, &P.row_jidx})
        for (int q : *v)
            if (q >= 0) ++placed[q];
    for (int k : placed) info[5] += k != 1;
    if (all_const) {
        for (size_t k = 0; k < P.jc_jidx.size(); ++k)
            if (P.jc_jidx[k] >= 0) faults += P.jc_val[k] != J.cval[P.jc_jidx[k]];
        for (size_t k = 1; k < P.jd.size(); k += 2) faults += P.jd[k] != -1;
        for (size_t k = 3; k < P.rows.size(); k += 4) faults += P.rows[k] != -1;
    }
    const int step = 2 * fsize * G;
    for (int c = 0; c < nrooms; ++c) {
        const int nlds = lds_pairs(P, (size_t)std::max(rooms[c], P.fixed_pairs));
        if (nlds < P.fixed_pairs || nlds > std::max(rooms[c], P.fixed_pairs)) ++faults;
        const int nspill = P.npairs - nlds, end = nlds * step;
        if (nspill == 0) continue;
        ++info[2];
        const BlockStreams S = build_block_streams(P, G, waves, fsize, nlds);
        // the pair at `off` for a lane that reads outside LDS, and `more` pairs behind it
        auto outside = [&](int off, int more) {
            const int q = std::max(off - end, 0);
            if (q % step || q / step + more >= nspill) ++faults;
        };
        auto whole = [&](int q) {  // the block at pair q lies on one side of the cut
            if (P.second[q + 1] && (q < nlds) != (q + 1 < nlds)) ++faults;
        };
        auto word = [&](int w) { return w & kBlkAddrMask; };
        for (int wv = 0; wv < waves; ++wv) {
            const size_t f1 = wv + 1 < waves ? (size_t)S.f_at[wv + 1] : S.fs.size() / 256;
            for (size_t u = S.f_at[wv]; u < f1; ++u) {
                const int* q = &S.fs[256 * u];
                const bool far = q[3] < 0;
                info[far ? 3 : 4]++;
                for (int k = 0; k < 64; ++k, q += 4) {
                    if ((q[3] < 0) != far) ++faults;
                    for (int x = 0; x < 3; ++x) {
                        whole(q[x] / step);
                        if (far) outside(q[x], 1);
                        else if (q[x] >= end) ++faults;
                    }
                    if (!(q[3] & kBlkEnd)) continue;
                    // the target's old value is read along by every lane of its team
                    const int to = q[3] & kBlkAssign ? P.zpair : word(q[3]);
                    whole(word(q[3]));
                    if (far) outside(to * step, 1);
                    else if (word(q[3]) >= nlds) ++faults;
                    if (q[3] & kBlkLead && q[3] & kBlkTwo && !P.second[word(q[3]) + 1]) ++faults;
                }
            }
            const size_t b1 = wv + 1 < waves ? (size_t)S.b_at[wv + 1] : S.bs.size() / 256;
            for (size_t u = S.b_at[wv]; u < b1; ++u) {
                const int* q = &S.bs[256 * u];
                for (int k = 0; k < 64; ++k, q += 4) {
                    whole(q[0] / step);
                    if (q[3] < 0 && !P.second[q[0] / step + 1]) ++faults;  // two columns: two pairs
                    for (int off : {q[0], q[0] + step, q[1]}) outside(off, 0);
                    if (!(q[3] & kBlkEnd)) continue;
                    whole(q[2] / step);
                    for (int off : {q[2], q[2] + step, word(q[3]) * step}) outside(off, 0);
                }
            }
        }
        // the dense phase reads LDS alone
        for (int x : P.tail_src) faults += x / 2 >= nlds;
    }
    return faults;
}

}  // extern "C"
