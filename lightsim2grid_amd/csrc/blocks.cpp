// Block plan of the factorisation and its lane streams (see blocks.hpp).
#include "blocks.hpp"

#include <algorithm>
#include <numeric>
#include <queue>
#include <stdexcept>
#include <string>

namespace pfgpu {

namespace {

int find_in(const std::vector<int>& v, int b, int e, int x) {
    const auto it = std::lower_bound(v.begin() + b, v.begin() + e, x);
    return it == v.begin() + e || *it != x ? -1 : (int)(it - v.begin());
}

// The buses with unknowns in elimination order, and the place of every unknown.
struct Buses {
    std::vector<int> bus;         // elimination position -> bus
    std::vector<int> w;           // its unknowns
    std::vector<int> blk, sub;    // J index -> elimination position, place in the block
    std::vector<int> pos;         // bus -> elimination position, -1
};

Buses order_buses(const JPattern& J, const std::vector<int>& perm) {
    const int npvpq = (int)J.pvpq.size(), off = J.off;
    auto bus_of = [&](int u) {
        if (off && u == 0) return J.slack0;
        const int k = u - off;
        return k < npvpq ? J.pvpq[k] : J.pq[k - npvpq];
    };
    Buses B;
    B.blk.assign(J.N, -1);
    B.sub.assign(J.N, 0);
    B.pos.assign(J.n_bus, -1);
    for (int u : perm) {
        const int b = bus_of(u);
        if (B.pos[b] < 0) {
            B.pos[b] = (int)B.bus.size();
            B.bus.push_back(b);
            B.w.push_back(0);
        }
        B.blk[u] = B.pos[b];
        B.sub[u] = B.w[B.pos[b]]++;
    }
    return B;
}

// Symbolic elimination tree of the symmetrised block pattern: arms[k] = rows below k, parent.
struct Arms {
    std::vector<int> cp, ci, parent;
};

Arms symbolic(int nb, std::vector<std::vector<int>>& low) {
    Arms A;
    A.cp.assign(nb + 1, 0);
    A.parent.assign(nb, -1);
    std::vector<std::vector<int>> arm(nb), child(nb);
    std::vector<int> mark(nb, -1);
    for (int k = 0; k < nb; ++k) {
        auto& s = arm[k];
        mark[k] = k;
        for (int r : low[k]) if (mark[r] != k) { mark[r] = k; s.push_back(r); }
        for (int c : child[k])
            for (int r : arm[c]) if (mark[r] != k) { mark[r] = k; s.push_back(r); }
        std::sort(s.begin(), s.end());
        if (!s.empty()) { A.parent[k] = s[0]; child[s[0]].push_back(k); }
        A.cp[k + 1] = A.cp[k] + (int)s.size();
    }
    A.ci.reserve(A.cp[nb]);
    for (auto& s : arm) A.ci.insert(A.ci.end(), s.begin(), s.end());
    return A;
}

// The smallest tail worth a dense phase of its own.
constexpr int kMinTail = 8;

// Pairs that the 160 KB of a CU's LDS hold at most (one instance in FP32).
constexpr int kMostUsed = 160 * 1024 / 8;

}  // namespace

bool has_block_form(const JPattern& J) { return J.rowpos.empty(); }
bool block_plan_fits(const BlockPlan& P) { return P.npairs < 1 << kBlkAddrBits; }

BlockPlan build_block_plan(const YbusPattern& Y, const JPattern& J, const std::vector<int>& perm, BlockOrder order) {
    if (order == kByLife) return by_life(build_block_plan(Y, J, perm, kByUse));
    BlockPlan P;
    const int n = Y.n, N = J.N;
    P.n = n;
    Buses B = order_buses(J, perm);
    const int nb = (int)B.bus.size();
    // block pattern of J: L side (row after column in the elimination order) and U side
    std::vector<std::vector<int>> lo(nb), up(nb), low(nb);  // lo[c]: rows; up[r]: columns
    for (int c = 0; c < N; ++c)
        for (int q = J.Jp[c]; q < J.Jp[c + 1]; ++q) {
            const int a = B.blk[J.Ji[q]], b = B.blk[c];
            if (a > b) lo[b].push_back(a);
            else if (a < b) up[a].push_back(b);
            if (a != b) low[std::min(a, b)].push_back(std::max(a, b));
        }
    const Arms A = symbolic(nb, low);
    // tail: the top chain of the elimination tree
    int k0 = nb, m = 0;
    while (k0 > 0 && (k0 == nb || A.parent[k0 - 1] == k0) && m + B.w[k0 - 1] <= kMaxTail) m += B.w[--k0];
    if (m < kMinTail) { k0 = nb; m = 0; }
    P.m = m;

    // exact pattern: a block of the symmetrised pattern is nonzero if J holds it or a product does
    const int na = A.cp[nb];
    std::vector<char> hasL(na, 0), hasU(na, 0), jL(na, 0), jU(na, 0);  // (of the tail too)
    for (int k = 0; k < nb; ++k) {
        for (int r : lo[k]) { const int q = find_in(A.ci, A.cp[k], A.cp[k + 1], r); hasL[q] = jL[q] = 1; }
        for (int c : up[k]) { const int q = find_in(A.ci, A.cp[k], A.cp[k + 1], c); hasU[q] = jU[q] = 1; }
    }
    // value ids: D(k) = k, y(k) = nb + k, L = 2 nb + q, U = 2 nb + na + q
    const int vL = 2 * nb, vU = 2 * nb + na, nv = 2 * nb + 2 * na;
    auto find_block = [&](int a, int b) {  // -1: not in the symmetrised pattern
        if (a == b) return a;
        const int k = std::min(a, b), q = find_in(A.ci, A.cp[k], A.cp[k + 1], std::max(a, b));
        return q < 0 ? -1 : (a > b ? vL : vU) + q;
    };
    auto id_of = [&](int a, int b) {
        const int id = find_block(a, b);
        if (id < 0) throw std::logic_error("pfgpu: a block outside the factor's pattern");
        return id;
    };
    struct Prod { int t, l, u, d; };
    std::vector<Prod> pr;
    std::vector<int> lis, uis;
    for (int k = 0; k < k0; ++k) {
        lis.clear();
        uis.clear();
        for (int q = A.cp[k]; q < A.cp[k + 1]; ++q) {
            if (hasL[q]) lis.push_back(q);
            if (hasU[q]) uis.push_back(q);
        }
        for (int ql : lis) {
            const int a = A.ci[ql];
            for (int qu : uis) {
                const int b = A.ci[qu], t = id_of(a, b);
                if (t >= vU) hasU[t - vU] = 1;
                else if (t >= vL) hasL[t - vL] = 1;
                pr.push_back({t, vL + ql, vU + qu, k});
            }
            pr.push_back({nb + a, vL + ql, nb + k, k});
        }
    }
    // products by target, levels in elimination order (a target's products come from earlier pivots)
    std::vector<int> cnt(nv + 1, 0);
    for (const Prod& p : pr) cnt[p.t + 1]++;
    for (int t = 0; t < nv; ++t) cnt[t + 1] += cnt[t];
    std::vector<int> at(cnt.begin(), cnt.end() - 1), by(pr.size());
    for (size_t i = 0; i < pr.size(); ++i) by[at[pr[i].t]++] = (int)i;
    std::vector<int> level(nv, 0);
    // products are listed by pivot: when pivot k's are reached, D(k), L(:, k), U(k, :) and y(k) have
    // received all of theirs
    for (const Prod& p : pr) level[p.t] = std::max(level[p.t], 1 + std::max({level[p.l], level[p.u], level[p.d]}));
    P.nlev = 0;
    for (int t = 0; t < nv; ++t) P.nlev = std::max(P.nlev, level[t]);
    // backward levels: x_j = D_j (y_j - sum U_ji x_i), the tail's solution first
    std::vector<int> bl(nb, -1);
    P.nblev = 0;
    for (int j = k0 - 1; j >= 0; --j) {
        int l = 0;
        for (int q = A.cp[j]; q < A.cp[j + 1]; ++q)
            if (hasU[q]) l = std::max(l, bl[A.ci[q]] + 1);
        bl[j] = l;
        P.nblev = std::max(P.nblev, l + 1);
    }

    // --- storage: zero pairs, then the recycled blocks and the right-hand sides / solutions ----------
    P.zpair = 0;
    int next = 2;
    std::vector<int> addr(nv, -1);
    struct Life { int id, t0, t1; long long acc; };
    std::vector<Life> one, two, rhs;
    std::vector<int> last(nv, -1);
    std::vector<long long> acc(nv, 0);
    for (const Prod& p : pr)
        for (int x : {p.l, p.u, p.d}) {
            last[x] = std::max(last[x], level[p.t]);
            ++acc[x];
        }
    for (int j = 0; j < k0; ++j) {
        const int t = P.nlev + 2 + bl[j];
        last[j] = std::max(last[j], t);
        ++acc[j];
        for (int q = A.cp[j]; q < A.cp[j + 1]; ++q)
            if (hasU[q]) { last[vU + q] = std::max(last[vU + q], t); ++acc[vU + q]; }
    }
    // the dense phase reads the tail's blocks after the last factor level
    for (int k = k0; k < nb; ++k) {
        last[k] = P.nlev + 1;
        for (int q = A.cp[k]; q < A.cp[k + 1]; ++q) last[vL + q] = last[vU + q] = P.nlev + 1;
    }
    for (int k = 0; k < nb; ++k) {
        two.push_back({k, 0, last[k], acc[k] + 2});
        for (int q = A.cp[k]; q < A.cp[k + 1]; ++q) {
            const int w = B.w[A.ci[q]];
            auto add = [&](int id, bool j) {
                const int t0 = j ? 0 : level[id];
                (w == 2 ? two : one).push_back({id, t0, std::max(last[id], t0), acc[id] + 2});
            };
            if (hasL[q]) add(vL + q, jL[q]);
            if (hasU[q]) add(vU + q, jU[q]);
        }
    }
    // right-hand sides and solutions (of a tail block: its solution) live all the time
    for (int j = 0; j < k0; ++j)
        for (int q = A.cp[j]; q < A.cp[j + 1]; ++q)
            if (hasU[q]) ++acc[nb + A.ci[q]];
    for (int k = 0; k < nb; ++k) rhs.push_back({nb + k, k, 1 << 30, acc[nb + k] + 4});
    // a block takes the place of one that was read for the last time before it is written (interval
    // colouring by size); places by decreasing accesses, so that a launch that cannot hold all of
    // them in LDS keeps the most used
    struct Place { int size; long long acc; bool fill, tail; int first; };  // fill: empty during the assembly
    auto in_tail = [&](int id) {
        if (id < 2 * nb) return id % nb >= k0;
        return (id < vU ? id - vL : id - vU) >= A.cp[k0];
    };
    std::vector<Place> places;
    std::vector<int> place_of(nv, -1);
    auto colour = [&](std::vector<Life>& v, int size) {
        std::stable_sort(v.begin(), v.end(), [](const Life& a, const Life& b) { return a.t0 < b.t0; });
        using E = std::pair<int, int>;
        std::priority_queue<E, std::vector<E>, std::greater<E>> free;
        for (const Life& x : v) {
            int p;
            if (!free.empty() && free.top().first < x.t0) {
                p = free.top().second;
                free.pop();
            } else {
                p = (int)places.size();
                places.push_back({size, 0, true, false, x.id});
            }
            place_of[x.id] = p;
            places[p].acc += x.acc;
            places[p].tail |= in_tail(x.id);
            if (x.t0 <= 0 || x.id >= nb && x.id < vL) places[p].fill = false;
            free.push({x.t1, p});
        }
    };
    colour(two, 2);
    colour(one, 1);
    colour(rhs, 1);
    std::vector<int> po(places.size());
    std::iota(po.begin(), po.end(), 0);
    std::stable_sort(po.begin(), po.end(), [&](int a, int b) {
        if (places[a].tail != places[b].tail) return places[a].tail;
        return places[a].acc * places[b].size > places[b].acc * places[a].size;
    });
    // Places that lie outside LDS in every launch: by the first column they serve, so that the blocks of a
    // column, which products read together, share cache lines. 10 000-bus N-1 in FP32, a workgroup's factor
    // levels 8.4 -> 6.9 ms and backward levels 2.5 -> 2.1. (By classes of use and column throughout, the FP64
    // 2000-bus N-1 loses what that gains: 1.63 -> 1.80 ms.)
    {
        auto column = [&](int p) {
            const int id = places[p].first;
            if (id < 2 * nb) return id % nb;
            const int q = id < vU ? id - vL : id - vU;
            return (int)(std::upper_bound(A.cp.begin(), A.cp.end(), q) - A.cp.begin()) - 1;
        };
        size_t first = 0;
        for (int pairs = next; first < po.size() && pairs < kMostUsed; ++first) pairs += places[po[first]].size;
        std::vector<int> col(places.size());
        for (size_t i = first; i < po.size(); ++i) col[po[i]] = column(po[i]);
        std::stable_sort(po.begin() + first, po.end(), [&](int a, int b) { return col[a] < col[b]; });
    }
    P.second.assign(next, 0);
    std::vector<int> at_of(places.size());
    for (int p : po) {
        P.places.push_back({next, places[p].size, places[p].acc, places[p].fill});
        at_of[p] = next;
        next += places[p].size;
        if (places[p].tail) P.fixed_pairs = next;
        P.second.push_back(0);
        if (places[p].size == 2) P.second.push_back(1);
    }
    for (int id = 0; id < nv; ++id)
        if (place_of[id] >= 0) addr[id] = at_of[place_of[id]];
    P.second.resize(next + 2, 0);
    P.fill_at = next;
    P.npairs = next + 1;  // a one-pair block's second pair is read (and not used)

    // --- target words -----------------------------------------------------------------------------
    auto word_of = [&](int a, int b) {  // block (a, b) of the factor
        const int in = a < b ? B.w[a] : B.w[b], out = a < b ? B.w[b] : B.w[a];
        return addr[id_of(a, b)] | (in == 2 ? kBlkIn2 : 0) | (out == 2 ? kBlkTwo : 0) | (a < b ? kBlkCols : 0);
    };
    auto word_y = [&](int a) { return addr[nb + a] | (B.w[a] == 2 ? kBlkIn2 : 0) | kBlkCols; };
    // --- factor tasks by level -----------------------------------------------------------------------
    std::vector<int> rowid(na), colid(na);
    for (int k = 0; k < nb; ++k)
        for (int q = A.cp[k]; q < A.cp[k + 1]; ++q) { rowid[q] = A.ci[q]; colid[q] = k; }
    std::vector<std::vector<int>> per(P.nlev + 1);
    for (int t = 0; t < nv; ++t)
        if (cnt[t + 1] > cnt[t]) per[level[t]].push_back(t);
    P.f_lvl.assign(1, 0);
    for (int l = 1; l <= P.nlev; ++l) {
        for (int t : per[l]) {
            int word;
            if (t < nb) word = word_of(t, t) | (t < k0 ? kBlkInv | kBlkTwo : 0);
            else if (t < vL) word = word_y(t - nb);
            else {
                const int q = t >= vU ? t - vU : t - vL;
                const int a = t >= vU ? colid[q] : rowid[q], b = t >= vU ? rowid[q] : colid[q];
                word = word_of(a, b);
                if (!(t >= vU ? jU[q] : jL[q])) word |= kBlkAssign;
            }
            P.tasks.push_back(word);
            P.tasks.push_back((int)P.prods.size() / 3);
            for (int i = cnt[t]; i < cnt[t + 1]; ++i) {
                const Prod& p = pr[by[i]];
                P.prods.push_back(addr[p.l]);
                P.prods.push_back(addr[p.u]);
                P.prods.push_back(addr[p.d]);
            }
            P.tasks.push_back((int)P.prods.size() / 3);
        }
        P.f_lvl.push_back((int)P.tasks.size() / 3);
    }
    // --- backward tasks ---------------------------------------------------------------------------
    std::vector<std::vector<int>> perb(P.nblev);
    for (int j = 0; j < k0; ++j) perb[bl[j]].push_back(j);
    P.b_lvl.assign(1, 0);
    for (int l = 0; l < P.nblev; ++l) {
        for (int j : perb[l]) {
            P.btasks.push_back(addr[nb + j]);
            P.btasks.push_back((int)P.bprods.size() / 3);
            for (int q = A.cp[j]; q < A.cp[j + 1]; ++q) {
                if (!hasU[q]) continue;
                P.bprods.push_back(addr[vU + q]);
                P.bprods.push_back(addr[nb + A.ci[q]]);
                P.bprods.push_back(B.w[A.ci[q]] == 2 ? 1 : 0);
            }
            P.btasks.push_back((int)P.bprods.size() / 3);
            P.btasks.push_back(addr[j]);
        }
        P.b_lvl.push_back((int)P.btasks.size() / 4);
    }
    // --- buses and tail ---------------------------------------------------------------------------------
    P.bus_y.assign(n, -1);
    for (int k = 0; k < nb; ++k) P.bus_y[B.bus[k]] = addr[nb + k] | (B.w[k] == 2 ? kBlkIn2 : 0);
    if (J.off) {
        P.slack_bus = J.slack0;
        P.slack_x = addr[nb + B.pos[J.slack0]];
    }
    for (int a = k0; a < nb; ++a)
        for (int r = 0; r < B.w[a]; ++r) {
            for (int b = k0; b < nb; ++b)
                for (int c = 0; c < B.w[b]; ++c) {
                    // the top chain of the elimination tree need not be dense
                    const int id = find_block(a, b);
                    const bool has = a == b || (id >= 0 && (a < b ? hasU[id - vU] : hasL[id - vL]));
                    P.tail_src.push_back(!has ? 2 * P.zpair : a < b ? 2 * (addr[id] + c) + r : 2 * (addr[id] + r) + c);
                }
            P.tail_src.push_back(2 * addr[nb + a] + r);
        }
    // --- J fill ------------------------------------------------------------------------------------------
    auto block_word = [&](int a, int b) {
        int word = word_of(a, b);
        if (a == b && a < k0 && cnt[a + 1] == cnt[a]) word |= kBlkInv | kBlkTwo;  // nothing to eliminate
        return word;
    };
    struct Const { int dst, j[4]; double v[4]; };
    std::vector<Const> consts;
    std::vector<int> cent(nv, -1), dst_of(Y.p[n], -1), jx((size_t)4 * Y.p[n], -1);
    for (int c = 0; c < N; ++c)
        for (int q = J.Jp[c]; q < J.Jp[c + 1]; ++q) {
            const int r = J.Ji[q], a = B.blk[r], b = B.blk[c];
            if (J.sel[q] == SEL_CONST) {
                const int id = id_of(a, b);
                if (cent[id] < 0) {
                    cent[id] = (int)consts.size();
                    consts.push_back({block_word(a, b), {-1, -1, -1, -1}, {0, 0, 0, 0}});
                }
                Const& k = consts[cent[id]];
                const int e = 2 * B.sub[r] + B.sub[c];
                k.j[e] = q;
                k.v[e] = J.cval[q];
                continue;
            }
            // the kernel computes the block from the Ybus entry: rows P, Q and columns Va, Vm
            int& d = dst_of[J.src[q]];
            if (d == -1) d = block_word(a, b);
            if (d != block_word(a, b) || B.sub[r] != (J.sel[q] & 1) || B.sub[c] != (J.sel[q] >> 1))
                throw std::runtime_error("pfgpu: a J entry lies outside its bus block");
            jx[4 * (size_t)J.src[q] + J.sel[q]] = q;
        }
    for (const Const& k : consts) {
        P.jc_dst.push_back(k.dst);
        P.jc_jidx.insert(P.jc_jidx.end(), k.j, k.j + 4);
        P.jc_val.insert(P.jc_val.end(), k.v, k.v + 4);
    }
    std::vector<std::vector<std::pair<int, int>>> per_row(n);  // {column, CSC position}, diagonal apart
    std::vector<int> diag(n, -1), order_rows;
    for (int c = 0; c < n; ++c)
        for (int q = Y.p[c]; q < Y.p[c + 1]; ++q) {
            if (Y.i[q] == c) diag[c] = q;
            else per_row[Y.i[q]].push_back({c, q});
        }
    for (int b = 0; b < n; ++b)
        if (P.bus_y[b] >= 0) order_rows.push_back(b);
    std::stable_sort(order_rows.begin(), order_rows.end(), [&](int a, int b) { return per_row[a].size() > per_row[b].size(); });
    for (int b : order_rows) {
        const int q = diag[b];
        P.rows.insert(P.rows.end(), {b, P.bus_y[b], q, dst_of[q]});
        P.row_len.push_back((int)per_row[b].size());
        P.row_jidx.insert(P.row_jidx.end(), &jx[4 * (size_t)q], &jx[4 * (size_t)q] + 4);
    }
    for (size_t k = 0; !order_rows.empty() && k < per_row[order_rows[0]].size(); ++k) {
        P.jd_ptr.push_back((int)P.jd_pos.size());
        for (int b : order_rows) {
            if (per_row[b].size() <= k) break;
            const auto [c, q] = per_row[b][k];
            P.jd.insert(P.jd.end(), {c, dst_of[q]});
            P.jd_pos.push_back(q);
            P.jd_jidx.insert(P.jd_jidx.end(), &jx[4 * (size_t)q], &jx[4 * (size_t)q] + 4);
        }
    }
    return P;
}

// The same places in another order: nothing but the pairs' names changes.
BlockPlan by_life(BlockPlan P) {
    std::vector<BlockPlan::Place> to = P.places;
    std::stable_sort(to.begin(), to.end(), [](const BlockPlan::Place& a, const BlockPlan::Place& b) {
        if (a.fill != b.fill) return b.fill;
        return a.acc * b.size > b.acc * a.size;
    });
    std::vector<int> name(P.npairs + 1, 0);
    int next = 2;  // after the zeros
    for (int q : {0, 1}) name[q] = q;
    P.second.assign(next, 0);
    P.fill_at = -1;
    for (auto& p : to) {
        if (p.fill && P.fill_at < 0) P.fill_at = next;
        for (int k = 0; k < p.size; ++k) {
            name[p.at + k] = next++;
            P.second.push_back(k == 1);
        }
        p.at = next - p.size;
    }
    name[next] = next;
    P.second.resize(next + 2, 0);
    if (P.fill_at < 0) P.fill_at = next;
    P.fixed_pairs = P.npairs;
    P.places = std::move(to);
    auto word = [&](int& w) {
        if (w != -1) w = (w & ~kBlkAddrMask) | name[w & kBlkAddrMask];
    };
    auto pair = [&](int& q) { q = name[q]; };
    auto each = [](std::vector<int>& v, size_t from, size_t step, auto f) {
        for (size_t i = from; i < v.size(); i += step) f(v[i]);
    };
    each(P.bus_y, 0, 1, word);
    if (P.slack_x >= 0) pair(P.slack_x);
    each(P.tail_src, 0, 1, [&](int& x) { x = 2 * name[x >> 1] + (x & 1); });
    each(P.rows, 1, 4, word);
    each(P.rows, 3, 4, word);
    each(P.jd, 1, 2, word);
    each(P.jc_dst, 0, 1, word);
    each(P.tasks, 0, 3, word);
    each(P.prods, 0, 1, pair);
    each(P.btasks, 0, 4, word);
    each(P.btasks, 3, 4, pair);
    each(P.bprods, 0, 3, pair);
    each(P.bprods, 1, 3, pair);
    return P;
}

int lds_pairs(const BlockPlan& P, size_t room) {
    if (room >= (size_t)P.npairs) return P.npairs;
    int q = (int)room;
    while (q > 0 && P.second[q]) --q;
    return q;
}

// ---------------------------------------------------------------------------
// Unit streams
// ---------------------------------------------------------------------------
namespace {

int log2_up(int x) {
    int l = 0;
    while ((1 << l) < x) ++l;
    return l;
}

// The chunks of one level: a chunk is one wave's worth of tasks that share a team size, `n` units each.
struct Chunk {
    int lt = 0, n = 1;
    std::vector<int> tasks;  // indices in the level
};

// Deals the tasks of a level (np products each) into chunks. Tasks go by decreasing team size, so that a
// chunk's teams are equal; a chunk keeps its first task's team size for the smaller ones that fill it up.
// n, the products of a lane, minimises an estimate of the level's time: the longer of one wave's chain
// (operand reads, products, the team's reduction, the target) and the issue of all waves of a SIMD.
std::vector<Chunk> deal_level(const std::vector<int>& np, int G, int waves) {
    const int width = std::max(1, 64 / G);  // lanes of one instance in a wave
    const int tmax = log2_up(width + 1) - 1;
    const int nt = (int)np.size();
    int maxnp = 1;
    for (int x : np) maxnp = std::max(maxnp, x);
    std::vector<int> ord(nt);
    std::iota(ord.begin(), ord.end(), 0);
    std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return np[a] > np[b]; });
    auto deal = [&](int n, auto chunk) {  // chunk(lt, units, first task, tasks)
        for (int i = 0; i < nt;) {
            const int p = np[ord[i]], lt = std::min(tmax, log2_up(std::max(1, (p + n - 1) / n)));
            const int m = std::min(width >> lt, nt - i);
            chunk(lt, std::max(1, (p + (1 << lt) - 1) >> lt), i, m);
            i += m;
        }
    };
    int best = 1;
    double best_cost = 1e300;
    for (int n = (maxnp + (1 << tmax) - 1) >> tmax; n <= maxnp; n = n < 16 ? n + 1 : n + n / 8) {
        double simd[4] = {0, 0, 0, 0}, chain = 0;
        int i = 0;
        deal(std::max(1, n), [&](int lt, int units, int, int) {
            simd[i++ % waves % 4] += 4.5 * (28.0 * units + 5.0 * lt + 50.0);
            chain = std::max(chain, 300.0 + 40.0 * units + 25.0 * lt);
        });
        const double issue = *std::max_element(simd, simd + 4);
        const double cost = std::max(chain, issue) + 0.1 * issue;
        if (cost < best_cost - 1e-9) {
            best_cost = cost;
            best = std::max(1, n);
        }
    }
    std::vector<Chunk> out;
    deal(best, [&](int lt, int units, int first, int m) {
        out.push_back({lt, units, std::vector<int>(ord.begin() + first, ord.begin() + first + m)});
    });
    return out;
}

// Lays the levels out: emit(task, product in the task or -1, last unit, unit) fills a lane's unit, which
// is preset to `pad`; close(units of 64 lanes) sees each finished one.
template <class NProds, class Emit, class Close>
void lay_levels(const std::vector<int>& lvl, int G, int waves, NProds nprods, Emit emit, Close close, const int (&pad)[4],
                std::vector<int>& out, std::vector<int>& at, std::vector<uint64_t>& mask, int& words) {
    const int nl = (int)lvl.size() - 1;
    words = std::max(1, (nl + 63) / 64);
    mask.assign((size_t)waves * words, 0);
    std::vector<std::vector<int>> ws(waves);
    for (int l = 0; l < nl; ++l) {
        const int t0 = lvl[l], nt = lvl[l + 1] - t0;
        std::vector<int> np(nt);
        for (int i = 0; i < nt; ++i) np[i] = nprods(t0 + i);
        const std::vector<Chunk> cs = deal_level(np, G, waves);
        for (size_t ci = 0; ci < cs.size(); ++ci) {
            const Chunk& c = cs[ci];
            const int w = (int)(ci % waves);
            std::vector<int>& st = ws[w];
            mask[(size_t)w * words + l / 64] |= 1ull << (l % 64);
            const int T = 1 << c.lt;
            for (int u = 0; u < c.n; ++u) {
                const bool end = u == c.n - 1;
                const size_t p = st.size();
                st.resize(p + 256);
                for (int k = 0; k < 64; ++k) std::copy(pad, pad + 4, &st[p + 4 * k]);
                for (size_t k = 0; k < c.tasks.size(); ++k)
                    for (int tp = 0; tp < T; ++tp) {
                        const int i = c.tasks[k], pi = u * T + tp;
                        int unit[4] = {pad[0], pad[1], pad[2], pad[3]};
                        emit(t0 + i, pi < np[i] ? pi : -1, end, end && tp == T - 1, unit);
                        for (int g = 0; g < G; ++g)
                            std::copy(unit, unit + 4, &st[p + 4 * ((k * T + tp) * G + g)]);
                    }
                int ctl = c.lt << kBlkTeamShift;
                if (end) ctl |= kBlkEnd;
                if (end && ci + waves >= cs.size()) ctl |= kBlkLevel;
                for (int k = 0; k < 64; ++k) st[p + 4 * k + 3] |= ctl;
                close(&st[p]);
            }
        }
    }
    at.assign(waves, 0);
    for (int w = 0; w < waves; ++w) {
        at[w] = (int)(out.size() / 256);
        if (w == 0) {
            size_t all = 0;
            for (const auto& s : ws) all += s.size() + 512 * kBlkAhead;
            out.reserve(all);
        }
        out.insert(out.end(), ws[w].begin(), ws[w].end());
        for (int k = 0; k < 64 * 2 * kBlkAhead; ++k) out.insert(out.end(), pad, pad + 4);
    }
    if (out.size() / 4 >= (size_t)1 << 31) throw std::runtime_error("pfgpu: block stream too large");
}

}  // namespace

BlockStreams build_block_streams(const BlockPlan& P, int G, int waves, int fsize, int nlds) {
    BlockStreams S;
    const int step = 2 * fsize * G;  // bytes between the pairs of one instance
    const int z = P.zpair * step, lds_end = nlds * step;
    const int pad[4] = {z, z, z, 0};
    if ((int64_t)P.npairs * step >= (int64_t)1 << 31) throw std::runtime_error("pfgpu: block stream offsets too large");
    auto none = [](int*) {};
    lay_levels(
        P.f_lvl, G, waves, [&](int t) { return P.tasks[3 * t + 2] - P.tasks[3 * t + 1]; },
        [&](int t, int pi, bool end, bool lead, int* w) {
            if (pi >= 0) {
                const int* p = &P.prods[3 * (P.tasks[3 * t + 1] + pi)];
                for (int k = 0; k < 3; ++k) w[k] = p[k] * step;
            }
            if (end) w[3] = P.tasks[3 * t] | (lead ? kBlkLead : 0);
        },
        [&](int* u) {
            bool wide = false;
            for (int k = 0; k < 64; ++k)
                wide |= u[4 * k] >= lds_end || u[4 * k + 1] >= lds_end || u[4 * k + 2] >= lds_end ||
                        ((u[4 * k + 3] & kBlkLead) && (u[4 * k + 3] & kBlkAddrMask) >= nlds);
            if (wide)
                for (int k = 0; k < 64; ++k) u[4 * k + 3] |= kBlkWide;
        },
        pad, S.fs, S.f_at, S.f_mask, S.f_words);
    lay_levels(
        P.b_lvl, G, waves, [&](int t) { return P.btasks[4 * t + 2] - P.btasks[4 * t + 1]; },
        [&](int t, int pi, bool end, bool lead, int* w) {
            if (pi >= 0) {
                const int* p = &P.bprods[3 * (P.btasks[4 * t + 1] + pi)];
                w[0] = p[0] * step;
                w[1] = p[1] * step;
                w[3] = p[2] ? kBlkWide : 0;
            }
            if (end) {
                w[2] = P.btasks[4 * t + 3] * step;
                w[3] |= P.btasks[4 * t] | (lead ? kBlkLead : 0);
            }
        },
        none, pad, S.bs, S.b_at, S.b_mask, S.b_words);
    return S;
}

}  // namespace pfgpu
